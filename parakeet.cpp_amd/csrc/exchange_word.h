// exchange_word.h -- words that workgroups wait for (constexpr: device code and host tests).
#pragma once

namespace pkdev {

// A word not written yet: the one f32 pattern (a NaN with every bit set) that no producer stores.
constexpr unsigned kEmpty = 0xffffffffu;
// A produced word: the empty pattern loses one payload bit and stays a NaN; any other is unchanged.
constexpr unsigned filled_word(unsigned b) { return b == kEmpty ? b - 1u : b; }
// Any of four words empty (the empty pattern is the largest).
constexpr bool any_empty(unsigned a, unsigned b, unsigned c, unsigned d) {
    const unsigned ab = a > b ? a : b, cd = c > d ? c : d;
    return (ab > cd ? ab : cd) == kEmpty;
}

}  // namespace pkdev
