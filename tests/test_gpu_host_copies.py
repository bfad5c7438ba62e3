"""Host-memory calls around the sizes where their copies change: frames up with the descriptor block in
one copy up to 1 MiB, outputs written straight into pinned memory up to 256 KiB (tokens, segments and
trace; the tapped logits too while all of them fit, and through pinned blocks of 4 MiB beyond).  On either
side of each line the results equal those of the same windows decoded from device frames with another
split of the outputs, bit for bit, and the logit rows of steps an utterance does not reach stay
untouched."""
import numpy as np
import pytest

from conftest import small_eou, small_tdt
from parity import check_window

pytestmark = pytest.mark.gpu

LINE_FRAMES, LINE_OUT = 1 << 20, 256 << 10


def _equal(a, b):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x["steps"] == y["steps"]
        for k in ("tokens", "segments", "ctrl"):
            assert np.array_equal(x[k], y[k]), k


@pytest.mark.parametrize("kind", ["tdt", "eou"])
@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_frames_line(tmp_path, kind, extra):
    from parakeet_amd import gguf, hipmem, pk, synth
    import oracle
    path = str(tmp_path / "d.gguf")
    (small_tdt if kind == "tdt" else small_eou)(path)
    om = oracle.OracleModel.from_gguf(path, gguf)
    dev = pk.Decoder.from_gguf(path, n_slots=64)
    D = dev.info.D
    rows = LINE_FRAMES // (4 * D) + extra
    T = [rows // 32] * 31
    T.append(rows - sum(T))
    encs = [synth.encoder_frames(40 + u, t, D) for u, t in enumerate(T)]
    print(f"{kind}: {rows} frames of {4 * D} bytes", flush=True)
    a = dev.decode(encs, slots=list(range(32)), trace=True)
    flat = hipmem.DeviceArray.from_numpy(np.concatenate(encs))
    first = np.concatenate([[0], np.cumsum(T)[:-1]])
    b = dev.decode_device_frames(flat.ptr, first, T, slots=list(range(32, 64)))
    _equal(a, b)
    check_window(om, dev, 0, encs[0], a[0], om.new_state(), dev.info.max_symbols)
    flat.free()
    dev.close()


@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_outputs_line(tmp_path, extra):
    from parakeet_amd import pk, synth
    path = str(tmp_path / "d.gguf")
    small_tdt(path)
    dev = pk.Decoder.from_gguf(path, n_slots=8)
    n, Vo = 4, dev.info.Vo
    encs = [synth.encoder_frames(60 + u, 3 + u, dev.info.D) for u in range(n)]
    steps = 64                                # more than any of the windows takes
    # words per utterance: tokens, segments (one more), logits
    cap = (LINE_OUT // 4 // n - 1 - steps * Vo) // 2 + extra
    print(f"token capacity {cap}", flush=True)
    a = dev.decode(encs, slots=[0, 1, 2, 3], token_cap=cap, logit_steps=steps)
    b = dev.decode(encs, slots=[4, 5, 6, 7])
    _equal(a, b)
    for x in a:
        assert 0 < x["steps"] < steps
        assert not np.isnan(x["logits"][:x["steps"]]).any()
        assert np.isnan(x["logits"][x["steps"]:]).all()
    dev.close()


# n sessions, tapped steps, frames of the first and of the others: the tap just past the pinned line with the
# tokens within it; several blocks of utterances (128 steps of 8,198 floats fit one); one utterance's steps in
# two blocks beside one of a few steps; tokens past the pinned line as well
@pytest.mark.parametrize("n,steps,first,rest,cap", [(8, 1, 3, 2, None), (150, 2, 2, 1, None), (2, 200, 120, 2, None),
                                                    (40, 3, 2, 3, 2000)])
def test_staged_tap(tmp_path, n, steps, first, rest, cap):
    from parakeet_amd import pk, synth
    path = str(tmp_path / "d.gguf")
    synth.make_shape(path, "tdt-0.6b-v3")
    dev = pk.Decoder.from_gguf(path, n_slots=n + 1)
    encs = [synth.encoder_frames(80 + u, first if u == 0 else rest, dev.info.D) for u in range(n)]
    print(f"{n} sessions, {steps} tapped steps", flush=True)
    got = dev.decode(encs, logit_steps=steps, token_cap=cap)
    assert max(x["steps"] for x in got) > 1
    for u in sorted({0, 1, n // 2, 126 % n, 127 % n, n - 1}):
        one = dev.decode([encs[u]], slots=[n], reset=[1], logit_steps=5)[0]   # into pinned memory by the kernel
        assert one["steps"] == got[u]["steps"] and np.array_equal(one["tokens"], got[u]["tokens"])
        k = min(steps, 5, one["steps"])
        a, b = got[u]["logits"][:k], one["logits"][:k]
        assert np.linalg.norm(a - b) <= 4e-6 * np.linalg.norm(b), u   # 32-bit sums in another order
        taken = min(steps, got[u]["steps"])
        assert not np.isnan(got[u]["logits"][:taken]).any() and np.isnan(got[u]["logits"][taken:]).all()
        # each tapped step's argmax is its decision: steps past the fifth are in their place too
        am = got[u]["logits"][:taken, :dev.info.V1].argmax(1)
        assert [t for t in am.tolist() if t != dev.info.blank] == got[u]["tokens"][:np.sum(am != dev.info.blank)].tolist()
    dev.close()
