"""Runs of blanks over the joint tile's spare columns.

A blank decision keeps the prediction output, so while an utterance is in a
run of blanks the joint's spare columns (a 16-column tile holds fewer
utterances than columns) evaluate its next frames in the same iteration, and
the decision step walks the run there.  The steps are the same joint
evaluations the one-step-per-iteration loop makes, so:

- every decision replays through the oracle (teacher-forced, zero unexplained
  mismatches, final state within 1e-3), TDT and EOU, blank-heavy decodes;
- tokens, steps, traces, segments and final state equal the loop with the runs
  turned off (PK_SPEC=0), bit for bit, while the iteration count drops;
- windows carried across calls give the same stream as one call."""
import os

import numpy as np
import pytest

from conftest import small_eou, small_tdt
from parity import check_window

pytestmark = pytest.mark.gpu


def _both(dev, encs, n, **kw):
    """The same decode with the runs on and off (fresh slots each)."""
    os.environ["PK_SPEC"] = "0"
    try:
        off = dev.decode(encs, slots=list(range(n, 2 * n)), trace=True, **kw)
        it_off = dev.last_timing()["iterations"]
    finally:
        os.environ.pop("PK_SPEC", None)
    on = dev.decode(encs, slots=list(range(n)), trace=True, **kw)
    it_on = dev.last_timing()["iterations"]
    return on, off, it_on, it_off


@pytest.mark.parametrize("B", [1, 2, 4, 40])
def test_tdt_blank_runs_replay_and_equal(tmp_path, B):
    """B=1 and B=2 run on one domain of every workgroup, whose keys one wave gathers while at
    most 2 joint columns are live and all eight waves once spare columns are in use; with the
    runs off every iteration takes the first form."""
    from parakeet_amd import gguf, pk, synth
    import oracle
    path = str(tmp_path / "m.gguf")
    small_tdt(path)
    dev = pk.Decoder.from_gguf(path, n_slots=2 * B)
    om = oracle.OracleModel.from_gguf(path, gguf)
    encs = [synth.encoder_frames(1200 + u, 60 - (u % 5) * 7, 128) for u in range(B)]
    bb = np.full(B, 3.0, np.float32)
    print(f"blank runs: TDT B={B}, blank +3", flush=True)
    on, off, it_on, it_off = _both(dev, encs, B, blank_bias=bb, max_symbols=10)
    for u in range(B):
        assert np.array_equal(on[u]["tokens"], off[u]["tokens"]), u
        assert np.array_equal(on[u]["trace"], off[u]["trace"]), u
        assert on[u]["steps"] == off[u]["steps"], u
        a, b = dev.read_state(u), dev.read_state(B + u)
        assert np.array_equal(a["h"], b["h"]) and np.array_equal(a["c"], b["c"]), u
        assert np.array_equal(a["ctrl"], b["ctrl"]), u
        check_window(om, dev, u, encs[u], on[u], om.new_state(), 10, blank_bias=3.0)
    assert it_on < it_off, (it_on, it_off)
    print(f"  iterations {it_on} with runs, {it_off} without", flush=True)
    dev.close()


def test_eou_blank_runs_replay_and_equal(tmp_path):
    from parakeet_amd import gguf, pk, synth
    import oracle
    path = str(tmp_path / "e.gguf")
    w = small_eou(path)
    bias = w["eou.joint.out.bias"].copy()
    bias[33] += 1.0   # <EOU> now and then, so resets interrupt the runs
    small_eou(path, overrides={"eou.joint.out.bias": bias})
    dev = pk.Decoder.from_gguf(path, n_slots=6)
    om = oracle.OracleModel.from_gguf(path, gguf)
    encs = [synth.encoder_frames(1300 + u, 50, 64) for u in range(3)]
    bb = np.full(3, 2.0, np.float32)
    on, off, it_on, it_off = _both(dev, encs, 3, blank_bias=bb, max_symbols=5)
    for u in range(3):
        for k in ("tokens", "trace", "segments"):
            assert np.array_equal(on[u][k], off[u][k]), (u, k)
        check_window(om, dev, u, encs[u], on[u], om.new_state(), 5, blank_bias=2.0)
    assert it_on < it_off, (it_on, it_off)
    dev.close()


def test_tdt_blank_runs_across_windows(tmp_path):
    """Windows of 7 frames with the state carried give the one-call stream (a run of
    blanks that reaches a window's end stops there and resumes in the next call)."""
    from parakeet_amd import pk, synth
    path = str(tmp_path / "m.gguf")
    small_tdt(path)
    dev = pk.Decoder.from_gguf(path, n_slots=2)
    enc = synth.encoder_frames(1400, 70, 128)
    bb = np.full(1, 3.0, np.float32)
    whole = dev.decode([enc], slots=[0], blank_bias=bb)[0]
    toks = []
    for t0 in range(0, 70, 7):
        toks += dev.decode([enc[t0:t0 + 7]], slots=[1], blank_bias=bb)[0]["tokens"].tolist()
    assert toks == whole["tokens"].tolist()
    dev.close()


def _lockstep(traces, T, durations, blank, max_symbols):
    """Joint columns of each lockstep iteration of one domain, from its utterances' decisions (T in
    the domain's order): one column per utterance with frames left, and the 16-column tile's spare
    ones dealt out evenly as later frames of the utterances whose last decision was a blank."""
    n = len(T)
    t, sym, step = [0] * n, [0] * n, [0] * n
    pend, keep = [True] * n, [False] * n
    cols = []
    while any(pend) or any(t[u] < T[u] for u in range(n)):
        live = [u for u in range(n) if t[u] < T[u]]
        spare = -len(live) % 16
        runs = [u for u in live if keep[u]] if spare else []
        ahead = [0] * n
        for i, u in enumerate(runs):
            q = spare // len(runs) + (1 if i < spare % len(runs) else 0)
            ahead[u] = min(q, T[u] - t[u] - 1)
        cols.append(len(live) + sum(ahead))
        pend = [False] * n
        for u in live:
            t0 = t[u]
            while True:
                tok, d = traces[u][step[u]]
                step[u] += 1
                dur = durations[d]
                keep[u] = tok == blank
                if tok == blank:
                    t[u], sym[u] = t[u] + max(1, dur), 0
                else:
                    pend[u], sym[u] = True, sym[u] + 1
                    if dur > 0 or sym[u] >= max_symbols:
                        t[u], sym[u] = t[u] + max(1, dur), 0
                if not keep[u] or t[u] >= T[u] or t[u] - t0 > ahead[u]:
                    break
    assert step == [len(x) for x in traces]
    return cols


@pytest.mark.parametrize("B,domains", [(1, 1), (2, 1), (5, 1), (20, 2), (40, 4)])
def test_key_gather_line(tmp_path, B, domains):
    """The argmax keys of an iteration are gathered by one wave while its loads cover every
    workgroup of the domain (P workgroups, column pairs rounded up to a power of two, P times pairs
    at most 256) and by all eight waves beyond.  Each launch here has iterations on both sides of
    that line, in an order that changes with the utterances' blanks; every decision replays
    through the oracle, its tapped logits included, and the iterations are those the decisions
    imply."""
    from parakeet_amd import gguf, pk, synth
    import oracle
    from parity import rel
    path = str(tmp_path / "m.gguf")
    small_tdt(path)
    dev = pk.Decoder.from_gguf(path, n_slots=B)
    om = oracle.OracleModel.from_gguf(path, gguf)
    P = pk.device_info()["n_cu"] // domains
    T = [70 - (u // domains) * 60 // max(1, (B - 1) // domains) for u in range(B)]   # ends one after the other
    encs = [synth.encoder_frames(1500 + u, T[u], 128) for u in range(B)]
    bb = np.array([(1.5, 0.0, 3.0)[(u // domains) % 3] for u in range(B)], np.float32)
    print(f"key gather: B={B} on {domains} domain(s) of {P}", flush=True)
    TAP = 40
    got = dev.decode(encs, trace=True, blank_bias=bb, max_symbols=5, logit_steps=TAP)
    iters = 0
    one_wave, all_waves = set(), set()
    order = sorted(range(B), key=lambda u: -T[u])   # longest first, dealt round robin
    for d in range(domains):
        us = order[d::domains]
        cols = _lockstep([got[u]["trace"].tolist() for u in us], [T[u] for u in us], [0, 1, 2, 3, 4], dev.info.blank, 5)
        iters = max(iters, len(cols))
        for c in cols:
            pairs = 1 if c <= 2 else 1 << ((c - 1).bit_length() - 1)
            if c:
                (one_wave if P * pairs <= 256 else all_waves).add(c)
    print(f"  columns gathered by one wave {sorted(one_wave)}, by all {sorted(all_waves)}", flush=True)
    assert one_wave and all_waves and min(all_waves) > max(one_wave)
    assert dev.last_timing()["iterations"] == iters
    for u in range(B):
        check_window(om, dev, u, encs[u], got[u], om.new_state(), 5, blank_bias=float(bb[u]))
        n = min(TAP, got[u]["steps"])
        rep = om.replay_window(encs[u], om.new_state(), 5, got[u]["trace"], blank_bias=float(bb[u]), n_tap=TAP)
        assert all(rel(got[u]["logits"][j], rep["logits"][j]) < 1e-3 for j in range(n)), u
    dev.close()


@pytest.mark.parametrize("B", [2, 4, 40])
def test_logit_tap_with_blank_runs(tmp_path, B):
    """The logit tap with the runs on: the joint logits of every step, including
    the steps a run takes from a spare column (possibly several frames ahead,
    after a duration skip), equal the oracle's logits of the same step within
    1e-3 (src/parakeet_tdt.cpp:154-177), and the bits equal the tap with the
    runs off."""
    from parakeet_amd import gguf, pk, synth
    import oracle
    from parity import rel
    path = str(tmp_path / "tdt06.gguf")
    synth.make_shape(path, "tdt-0.6b-v3")
    dev = pk.Decoder.from_gguf(path, n_slots=2 * B)
    om = oracle.OracleModel.from_gguf(path, gguf)
    encs = [synth.encoder_frames(1300 + u, 40 + 3 * (u % 4), 1024) for u in range(B)]
    bb = np.full(B, 4.0, np.float32)
    TAP = 64
    print(f"logit tap with blank runs: TDT-0.6b B={B}, blank +4, {TAP} steps", flush=True)
    on, off, it_on, it_off = _both(dev, encs, B, blank_bias=bb, max_symbols=10, logit_steps=TAP)
    assert it_on < it_off, (it_on, it_off)           # the runs were taken
    worst = 0.0
    for u in range(B):
        assert np.array_equal(on[u]["trace"], off[u]["trace"]), u
        n = min(TAP, on[u]["steps"])
        assert np.array_equal(on[u]["logits"][:n], off[u]["logits"][:n]), u
        rep = om.replay_window(encs[u], om.new_state(), 10, on[u]["trace"], blank_bias=4.0, n_tap=TAP)
        assert rep["stats"]["unexplained"] == 0, rep["stats"]
        for j in range(n):
            worst = max(worst, rel(on[u]["logits"][j], rep["logits"][j]))
    assert worst < 1e-3, worst
    print(f"  iterations {it_on} (runs on) vs {it_off}; worst logit rel {worst:.2e}", flush=True)
