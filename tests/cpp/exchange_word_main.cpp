// Host-only driver of csrc/exchange_word.h: every NaN pattern, the edges around them and a spread of
// other words go through filled_word and any_empty.  Prints the number of patterns checked.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <initializer_list>

#include "exchange_word.h"

using pkdev::any_empty;
using pkdev::filled_word;
using pkdev::kEmpty;

namespace {

float as_float(unsigned b) {
    float f;
    memcpy(&f, &b, 4);
    return f;
}

bool check(unsigned b) {
    const unsigned w = filled_word(b);
    if (w == kEmpty) return false;                                        // a consumer would wait for it
    if (w != b && (b != kEmpty || !std::isnan(as_float(w)))) return false;   // changed: only the empty NaN, into a NaN
    const unsigned x[4][4] = {{b, 0, 0, 0}, {0, b, 0, 0}, {0, 0, b, 0}, {0, 0, 0, b}};
    for (const auto &v : x) {
        if (any_empty(v[0], v[1], v[2], v[3]) != (b == kEmpty)) return false;
        if (any_empty(filled_word(v[0]), filled_word(v[1]), filled_word(v[2]), filled_word(v[3]))) return false;
    }
    return true;
}

}  // namespace

int main() {
    long n = 0;
    const auto run = [&](unsigned b) {
        ++n;
        if (!check(b)) printf("0x%08x\n", b);
        return check(b);
    };
    if (!std::isnan(as_float(kEmpty))) return 1;
    for (unsigned sign : {0u, 0x80000000u})
        for (unsigned m = 0; m <= 0x7fffffu; ++m)          // infinity, then every NaN of the sign
            if (!run(sign | 0x7f800000u | m)) return 1;
    for (unsigned b = 0; b < 0xffff0000u; b += 65521u)     // numbers of every size
        if (!run(b)) return 1;
    // an empty word beside any other, in every place
    for (unsigned other : {0u, 1u, 0x7f800000u, 0x7fc00000u, 0x80000000u, 0xff800000u, 0xffc00000u, 0xfffffffeu, kEmpty})
        if (!any_empty(kEmpty, other, other, other) || !any_empty(other, kEmpty, other, other) ||
            !any_empty(other, other, kEmpty, other) || !any_empty(other, other, other, kEmpty))
            return 1;
    printf("%ld\n", n);
    return 0;
}
