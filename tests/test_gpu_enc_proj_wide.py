"""The enc_proj kernel of large batches (128 x 320 tiles) against the one-wave-per-block kernel: equal
bit for bit in every step's logits, for each storage of W_e (block integers and scales, f16, f32 hi and
lo), at the edges of its tiles: fewer rows than a tile, one more than a tile, a row block past the eighth
(workgroups are numbered in groups of eight row blocks), joint widths below, at and past one column block.
The first utterances are replayed through the oracle."""
import numpy as np
import pytest

from parity import check_window
from test_gpu_enc_proj import _run, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quant", ["q8_0", "q4_0", "f16", "f32"])
@pytest.mark.parametrize("J", [64, 320, 352])
@pytest.mark.parametrize("rows", [5, 128, 129, 1153])
def test_wide_enc_proj(tmp_path, quant, J, rows):
    from parakeet_amd import gguf, pk, synth
    import oracle
    path = str(tmp_path / "d.gguf")
    synth.make_decoder_gguf(path, kind="tdt", H=64, L=1, J=J, D=96, vocab=63, durations=[0, 1, 2], quant=quant)
    om = oracle.OracleModel.from_gguf(path, gguf)
    Ts = [rows] if rows < 8 else [3, 1, rows // 2, rows - 4 - rows // 2]   # ragged: tiles shared by utterances
    dev = pk.Decoder.from_gguf(path, n_slots=2 * len(Ts))
    encs = [synth.encoder_frames(700 + u, T, dev.info.D) for u, T in enumerate(Ts)]
    print(f"wide enc_proj, {quant} J={J} rows={rows}", flush=True)
    steps = 3 * max(Ts)
    a = _run(dev, encs, 0, "wide", logit_steps=steps)
    b = _run(dev, encs, len(Ts), "narrow", logit_steps=steps)
    _same(dev, a, b, len(Ts), 0, len(Ts))
    for u in range(min(2, len(Ts))):
        check_window(om, dev, u, encs[u], a[u], om.new_state(), 10)
    dev.close()
