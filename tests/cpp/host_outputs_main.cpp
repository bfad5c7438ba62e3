// Host-only driver of csrc/host_outputs.h (built with AddressSanitizer + UBSan): what a decode call
// copies into the caller's arrays after a launch, with counters a failed launch left stale and with
// those of a finished one.  Prints "ok".
#include <climits>
#include <cstdio>
#include <vector>

#include "host_outputs.h"

#define CHECK(x) do { if (!(x)) { fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #x); return 1; } } while (0)

namespace {

constexpr int kN = 4, kM = 3, kTok = 5, kSeg = 3, kTr = 4, kSteps = 2, kVo = 7;

struct Caller {   // 4 utterances, of which the launch ran 2, 0 and 3 (in this order)
    std::vector<int32_t> tok = std::vector<int32_t>(kN * kTok, -7), seg = std::vector<int32_t>(kN * kSeg, -7),
                         tr = std::vector<int32_t>(kN * kTr * 2, -7), ctrl = std::vector<int32_t>(kN * PK_CTRL_N, -7),
                         n_tok = std::vector<int32_t>(kN, 0), steps = std::vector<int32_t>(kN, 0),
                         n_seg = std::vector<int32_t>(kN, 0);
    std::vector<float> logits = std::vector<float>(kN * kSteps * kVo, -7.f);
    std::vector<int> map{2, 0, 3};
    pk_batch bt{};
    Caller() {
        bt.n_utts = kN;
        bt.tokens = tok.data();
        bt.token_cap = kTok;
        bt.n_tokens = n_tok.data();
        bt.steps = steps.data();
        bt.segments = seg.data();
        bt.seg_cap = kSeg;
        bt.n_segments = n_seg.data();
        bt.trace = tr.data();
        bt.trace_cap = kTr;
        bt.ctrl_out = ctrl.data();
        bt.logits = logits.data();
        bt.logit_steps = kSteps;
    }
    pkhost::HostOutputs outputs() {
        pkhost::HostOutputs o;
        o.bt = &bt;
        o.map = map.data();
        o.m = kM;
        o.tcap = kTok;
        o.scap = kSeg;
        o.trcap = kTr;
        o.lsteps = kSteps;
        o.Vo = kVo;
        return o;
    }
    bool untouched() const {
        for (const auto *v : {&tok, &seg, &tr, &ctrl})
            for (int32_t x : *v)
                if (x != -7) return false;
        for (const auto *v : {&n_tok, &steps, &n_seg})
            for (int32_t x : *v)
                if (x != 0) return false;
        for (float x : logits)
            if (x != -7.f) return false;
        return true;
    }
};

// A launch's staging rows: row i of each output counts up from 100 * (i + 1).
struct Staged {
    std::vector<int> tok, seg, tr;
    std::vector<int32_t> ctrl;
    std::vector<float> logits;
    Staged(int wt, int ws, int wr) {
        for (int i = 0; i < kM; ++i) {
            for (int k = 0; k < wt; ++k) tok.push_back(100 * (i + 1) + k);
            for (int k = 0; k < ws; ++k) seg.push_back(100 * (i + 1) + k);
            for (int k = 0; k < 2 * wr; ++k) tr.push_back(100 * (i + 1) + k);
            for (int k = 0; k < PK_CTRL_N; ++k) ctrl.push_back(100 * (i + 1) + k);
            for (int k = 0; k < kSteps * kVo; ++k) logits.push_back(float(100 * (i + 1) + k));
        }
    }
};

// ks, us: tapped steps and utterances staged at a time (0: all in place)
void copy_back(const pkhost::HostOutputs &o, const Staged &s, int wt, int ws, int wr, int ks, int us) {
    o.place(s.tok.data(), wt, s.seg.data(), ws, s.tr.data(), wr, s.ctrl.data());
    if (ks == 0) return o.place_tap(s.logits.data(), 0, kM, 0, kSteps);
    const int wide = o.widest(&pkhost::HostOutputs::tapped);
    for (int k0 = 0; k0 < wide; k0 += ks)
        for (int i0 = 0; i0 < kM; i0 += us) {
            const int nk = std::min(ks, wide - k0), i1 = std::min(kM, i0 + us);
            std::vector<float> rows;
            for (int i = i0; i < i1; ++i)
                for (int k = 0; k < nk * kVo; ++k) rows.push_back(s.logits[((size_t)i * kSteps + k0) * kVo + k]);
            o.place_tap(rows.data(), i0, i1, k0, nk);
        }
}

// Counters that a failed launch left as an earlier call's words: a trace's -1, logit bits, capacities.
int failed_launch() {
    const int words[] = {-1, INT_MIN, INT_MAX, 0x3f800000, (int)0xbf800000u, kTok, 1 << 20};
    for (int code : {PK_ERR_TIMEOUT, PK_ERR_DEVICE})
        for (int w : words) {
            Caller c;
            pkhost::HostOutputs o = c.outputs();
            const int status[4] = {code, 0, 0, 0};
            const std::vector<int> counters(3 * kM, w);
            CHECK(o.accept(status, counters.data()) == code);
            CHECK(o.widest(&pkhost::HostOutputs::tokens) == 0 && o.widest(&pkhost::HostOutputs::segments) == 0);
            CHECK(o.widest(&pkhost::HostOutputs::traced) == 0 && o.widest(&pkhost::HostOutputs::tapped) == 0);
            copy_back(o, Staged(kTok, kSeg, kTr), kTok, kSeg, kTr, 0, 0);
            CHECK(c.untouched());
        }
    return 0;
}

// A finished launch: counters within and past the capacities, rows at full capacity and as prefixes,
// the tap in place and staged in parts.
int finished_launch() {
    const std::vector<int> counters{3, 9, 0, /* steps */ 2, 6, 0, /* segments */ 1, 4, 0};
    const int status[4] = {0, 11, PK_ERR_OVERFLOW, 0};
    const int stages[][2] = {{0, 0}, {1, 1}, {1, 2}, {2, 1}, {2, 2}, {2, 3}};
    for (const auto &stage : stages) {
        const bool prefix = stage[0] != 0;
        Caller c;
        pkhost::HostOutputs o = c.outputs();
        CHECK(o.accept(status, counters.data()) == 0);
        const int wt = prefix ? o.widest(&pkhost::HostOutputs::tokens) : kTok,
                  ws = prefix ? o.widest(&pkhost::HostOutputs::segments) : kSeg,
                  wr = prefix ? o.widest(&pkhost::HostOutputs::traced) : kTr;
        CHECK(wt == kTok && ws == kSeg && wr == kTr);
        copy_back(o, Staged(wt, ws, wr), wt, ws, wr, stage[0], stage[1]);
        for (int u = 0; u < kN; ++u) {
            const int i = u == 2 ? 0 : u == 0 ? 1 : u == 3 ? 2 : -1;   // the launch's index of utterance u
            const int nt = i < 0 ? 0 : counters[i], ns = i < 0 ? 0 : counters[kM + i], ng = i < 0 ? 0 : counters[2 * kM + i];
            CHECK(c.n_tok[u] == nt && c.steps[u] == ns && c.n_seg[u] == ng);
            for (int k = 0; k < kTok; ++k) CHECK(c.tok[u * kTok + k] == (k < nt ? 100 * (i + 1) + k : -7));
            for (int k = 0; k < kSeg; ++k) CHECK(c.seg[u * kSeg + k] == (k < ng ? 100 * (i + 1) + k : -7));
            for (int k = 0; k < 2 * kTr; ++k) CHECK(c.tr[u * kTr * 2 + k] == (k < 2 * ns ? 100 * (i + 1) + k : -7));
            for (int k = 0; k < PK_CTRL_N; ++k) CHECK(c.ctrl[u * PK_CTRL_N + k] == (i >= 0 ? 100 * (i + 1) + k : -7));
            for (int k = 0; k < kSteps * kVo; ++k)
                CHECK(c.logits[u * kSteps * kVo + k] == (k < ns * kVo ? float(100 * (i + 1) + k) : -7.f));
        }
    }
    return 0;
}

}  // namespace

int main() {
    if (failed_launch() || finished_launch()) return 1;
    puts("ok");
    return 0;
}
