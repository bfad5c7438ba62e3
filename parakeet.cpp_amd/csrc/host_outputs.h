// host_outputs.h -- how a finished launch's results reach the caller's host arrays (host code only).
#pragma once

#include <algorithm>
#include <cstdint>
#include <cstring>

#include "parakeet_hip.h"

namespace pkhost {

// A launch's results in staging rows; utterance i of the launch is utterance map[i] of the batch.
// The counters (n_tokens, steps, n_segments, m each) give the lengths of what is copied.  A launch
// that ended with an error has written none of them, and their place holds whatever it held before:
// accept() takes them only from a launch without an error, and until then every length is 0.
struct HostOutputs {
    const pk_batch *bt = nullptr;
    const int *map = nullptr;
    int m = 0;
    int tcap = 0, scap = 0, trcap = 0;   // row capacities; scap: 0 without bt->segments, trcap: 0 without bt->trace
    int lsteps = 0, Vo = 0;              // tapped steps and floats of one (lsteps 0: no tap)
    const int *n_tok = nullptr, *n_steps = nullptr, *n_seg = nullptr;

    // status[0]: the launch's error word.  Returns it.
    int accept(const int *status, const int *counters) {
        if (status[0] != 0) return status[0];
        n_tok = counters;
        n_steps = counters + m;
        n_seg = counters + 2 * (size_t)m;
        return 0;
    }
    static int clamp(int n, int cap) { return std::max(0, std::min(n, cap)); }
    int tokens(int i) const { return n_tok ? clamp(n_tok[i], tcap) : 0; }
    int segments(int i) const { return n_seg ? clamp(n_seg[i], scap) : 0; }
    int traced(int i) const { return n_steps ? clamp(n_steps[i], trcap) : 0; }
    int tapped(int i) const { return n_steps ? clamp(n_steps[i], lsteps) : 0; }
    template <class Fn>
    int widest(Fn len) const {   // longest row of the launch, len one of the four above
        int w = 0;
        for (int i = 0; i < m; ++i) w = std::max(w, (this->*len)(i));
        return w;
    }

    // Rows of width wt / ws / wr (trace: pairs) at tok / seg / tr, and the control words (nullable).
    void place(const int *tok, int wt, const int *seg, int ws, const int *tr, int wr, const int32_t *ctrl) const {
        if (!n_tok) return;
        for (int i = 0; i < m; ++i) {
            const size_t u = (size_t)map[i];
            bt->n_tokens[u] = n_tok[i];
            bt->steps[u] = n_steps[i];
            if (bt->n_segments) bt->n_segments[u] = n_seg[i];
            if (const int n = tokens(i)) memcpy(bt->tokens + u * tcap, tok + (size_t)i * wt, 4 * (size_t)n);
            if (const int n = segments(i)) memcpy(bt->segments + u * scap, seg + (size_t)i * ws, 4 * (size_t)n);
            if (const int n = traced(i)) memcpy(bt->trace + u * trcap * 2, tr + (size_t)i * wr * 2, 8 * (size_t)n);
            if (ctrl) memcpy(bt->ctrl_out + u * PK_CTRL_N, ctrl + (size_t)i * PK_CTRL_N, PK_CTRL_N * 4);
        }
    }
    // Tapped steps k0 .. k0 + nk - 1 of utterances i0 .. i1 - 1, rows of nk steps at `rows`: those taken.
    void place_tap(const float *rows, int i0, int i1, int k0, int nk) const {
        for (int i = i0; i < i1; ++i) {
            const int n = clamp(tapped(i) - k0, nk);
            if (n > 0)
                memcpy(bt->logits + ((size_t)map[i] * lsteps + k0) * Vo, rows + (size_t)(i - i0) * nk * Vo,
                       (size_t)n * Vo * 4);
        }
    }
};

}  // namespace pkhost
