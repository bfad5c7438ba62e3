"""The word-by-word exchange between the workgroups of a domain, at the edges of its row and
column capacities: list rows staged 4 or 16 to a tile (lists of 4 and 5), row capacities of 8, 16
and 32 (8, 9, 16, 17 utterances per domain), key columns read in pairs (1, 2, 3 columns), duration
keys on one rank or two.  Two windows per utterance (state carried from the first), every step
replayed through the oracle; a blank offset on some utterances leaves spare columns in use."""
import numpy as np
import pytest

from parity import check_window

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 2, 3, 4, 5, 8, 9, 16, 17, 33, 64, 257, 272, 273])
@pytest.mark.parametrize("vocab", [95, 90])   # duration rows in one 16-row tile, across two
def test_exchange_capacities(tmp_path, B, vocab):
    from parakeet_amd import gguf, pk, synth
    import oracle
    path = str(tmp_path / "d.gguf")
    synth.make_decoder_gguf(path, kind="tdt", H=96, L=2, J=160, D=64, vocab=vocab, durations=[0, 1, 2, 3, 4, 5, 6, 8],
                            quant="q8_0")
    om = oracle.OracleModel.from_gguf(path, gguf)
    dev = pk.Decoder.from_gguf(path, n_slots=B)
    print(f"B={B} vocab={vocab}", flush=True)
    pick = range(B) if B <= 17 else sorted({0, 1, B // 2, B - 1, *range(3, B, B // 12)})
    states = {u: om.new_state() for u in pick}
    off = np.array([(0.0, 0.0, 2.0)[u % 3] for u in range(B)], np.float32)
    for window in range(2):
        encs = [synth.encoder_frames(9000 + 1000 * window + u, 9 + (5 * u) % 7, 64) for u in range(B)]
        res = dev.decode(encs, trace=True, blank_bias=off)
        for u in pick:
            check_window(om, dev, u, encs[u], res[u], states[u], 10, blank_bias=float(off[u]))
    dev.close()
