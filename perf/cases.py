"""Performance cases of the transducer greedy decode, through the public Python binding (parakeet_amd.pk).

A case is one caller's pass over a batch of sessions: `calls` consecutive decode windows of `frames`
encoder frames each (or ragged lengths from `frames_lo` to `frames`), the state carried from window to
window on the device, the first one from a fresh state, and then one short window more (TAIL frames)
whose first step also returns its joint logits (a single session's LSTM state is read back as well).
Offline transcription is one long window; live captioning is many two-frame chunks.

The decoders have the published shapes (synth.SHAPES) and dense random weights, with structure added
where a trained transducer has it: the output row of a token and its embedding share a direction, the
prediction network favours what it has not just emitted, and the frames carry token, blank and duration
evidence.  Decoding then runs as it does on speech: a token on about every second step, blanks between,
durations of 0 to 4 frames, silences, clear decisions (the best logit stands several units above the
next).  A program's results do not hang on the last bits of its logits, and neither do these.
"""
import os
import tempfile

import numpy as np
import torch

import __graft_entry__ as _entry

_entry.load_package()
from parakeet_amd import pk, synth  # noqa: E402

TAIL = 5            # frames of the last window: more than any duration carries over
N_SLOTS = 512       # sessions one decoder holds: the largest batch of a call
CHUNK = 65536       # frame rows made at once
A_TOK, A_BLANK, A_DUR, A_AFTER = 2.0, 1.8, 0.9, 1.0   # evidence in a frame: token, blank, duration, blank under a token
TOKEN_DURATIONS = (0.05, 0.25, 0.30, 0.20, 0.20)      # of a TDT token, 0 .. 4 frames
BLANK_DURATIONS = (0.0, 0.30, 0.25, 0.20, 0.25)       # of a TDT blank


def listed():
    return [
        # one live session: two-frame chunks as they arrive, frames and results in host memory
        dict(name="eou120m_live_1", shape="eou-120m", quant="q8_0", sessions=1, frames=2, calls=8,
             host=True, speech=0.7, offsets=False),
        # one 10 s utterance from the command line, frames and results in host memory
        dict(name="tdt06b_file_1x125", shape="tdt-0.6b-v3", quant="q8_0", sessions=1, frames=125, calls=1,
             host=True, speech=0.8, offsets=False),
        # one 2 min recording, decoded where the encoder left it
        dict(name="tdt06b_long_1x1501", shape="tdt-0.6b-v3", quant="q8_0", sessions=1, frames=1501, calls=1,
             host=False, speech=0.8, offsets=False),
        # a few utterances of uneven length in one request, 5-bit weights
        dict(name="tdt06b_q5_ragged_7", shape="tdt-0.6b-v3", quant="q5_0", sessions=7, frames=331, frames_lo=40,
             calls=1, host=True, speech=0.8, offsets=False),
        # a small server batch of 24 s segments, f16 weights
        dict(name="tdt11b_f16_24x301", shape="tdt-1.1b", quant="f16", sessions=24, frames=301, calls=1,
             host=False, speech=0.8, offsets=False),
        # a turn-taking model over finished recordings
        dict(name="eou120m_f16_16x375", shape="eou-120m", quant="f16", sessions=16, frames=375, calls=1,
             host=True, speech=0.7, offsets=False),
        # 128 live sessions, two-frame chunks, states carried, frames on the device
        dict(name="eou120m_live_128", shape="eou-120m", quant="q8_0", sessions=128, frames=2, calls=20,
             host=False, speech=0.7, offsets=False),
        # a batch of one-minute utterances
        dict(name="tdt06b_64x750", shape="tdt-0.6b-v3", quant="q8_0", sessions=64, frames=750, calls=1,
             host=False, speech=0.8, offsets=False),
        # a large batch of half-minute utterances, f16 weights
        dict(name="tdt11b_f16_256x375", shape="tdt-1.1b", quant="f16", sessions=256, frames=375, calls=1,
             host=False, speech=0.8, offsets=False),
        # a large batch of one-minute utterances
        dict(name="tdt06b_256x750", shape="tdt-0.6b-v3", quant="q8_0", sessions=256, frames=750, calls=1,
             host=False, speech=0.8, offsets=False),
        # a full batch of 4 s to 2 min utterances, blank offsets of 0, 2 and 4
        dict(name="tdt06b_ragged_512", shape="tdt-0.6b-v3", quant="q8_0", sessions=512, frames=1500, frames_lo=50,
             calls=1, host=False, speech=0.8, offsets=True),
    ]


def draw(rng):
    shape = rng.choice(["tdt-0.6b-v3", "tdt-0.6b-v3", "tdt-1.1b", "eou-120m"])
    quant = rng.choice({"tdt-0.6b-v3": ["q8_0", "q8_0", "q8_0", "q5_0", "q4_0"], "tdt-1.1b": ["f16", "f16", "q8_0", "f32"],
                        "eou-120m": ["q8_0", "q8_0", "f16"]}[shape])
    sessions = int(round(512 ** rng.random()))
    live = shape == "eou-120m" and rng.random() < 0.6
    case = dict(shape=shape, quant=quant, sessions=sessions)
    if live:
        case.update(frames=rng.randint(1, 9), calls=rng.randint(4, 24))
    else:
        most = min(1500, 300000 // sessions)
        frames = max(20, int(round(20 * (most / 20) ** rng.random())))
        case.update(frames=frames, calls=1)
        if sessions > 1 and rng.random() < 0.5:
            case["frames_lo"] = max(TAIL, int(frames * rng.uniform(0.03, 0.8)))
    case["host"] = sessions * case["frames"] <= 6000 and rng.random() < 0.5
    case["speech"] = round(rng.uniform(0.4, 0.95), 2)
    case["offsets"] = shape != "eou-120m" and rng.random() < 0.3
    return case


# ---------------------------------------------------------------- decoders

_models = {}


class _Model:
    """One decoder checkpoint, opened once for the life of the program."""

    def __init__(self, shape, quant):
        cfg = synth.SHAPES[shape]
        H, J, D, L, V1 = cfg["H"], cfg["J"], cfg["D"], cfg["L"], cfg["vocab"] + 1
        n_dur = len(cfg.get("durations", []))
        rng = np.random.default_rng(20240607)

        def normal(*s):
            return rng.standard_normal(s, dtype=np.float32)

        p = cfg["kind"]
        z = normal(V1 + n_dur, J)              # direction of each output row
        over = {f"{p}.predict.embed.weight": 0.6 * z[:V1], f"{p}.joint.out.weight": z / np.sqrt(J)}
        for l in range(L):
            w = 0.5 * normal(4 * H, H) / np.sqrt(H)
            w[2 * H:3 * H] += np.eye(H, dtype=np.float32)
            over[f"{p}.predict.lstm.{l}.w_ih"] = w.astype(np.float32)
            over[f"{p}.predict.lstm.{l}.w_hh"] = (0.5 * normal(4 * H, H) / np.sqrt(H)).astype(np.float32)
            b = 0.1 * normal(4 * H)
            b[:H] += 2.0                       # input gate open, forget gate mostly closed, output gate open
            b[H:2 * H] -= 1.0
            b[3 * H:] += 2.0
            over[f"{p}.predict.lstm.{l}.b_ih"] = b
        gain = 5.0 if L == 1 else 6.5
        over[f"{p}.joint.pred.weight"] = (0.3 * normal(J, H) / np.sqrt(H) - gain * np.eye(J, H)).astype(np.float32)
        with tempfile.TemporaryDirectory() as tmp:
            path = os.path.join(tmp, "decoder.gguf")
            self.w = synth.make_shape(path, shape, quant=quant, overrides=over)
            self.dec = pk.Decoder.from_gguf(path, n_slots=N_SLOTS)
        self.dec.set_timing(False)
        self.cfg, self.info, self.prefix = cfg, self.dec.info, p
        self.z = torch.from_numpy(z).cuda()
        w_e = torch.from_numpy(self.w[f"{p}.joint.enc.weight"]).double()
        self.pinv = torch.linalg.pinv(w_e).T.contiguous().float().cuda()      # [J, D]
        self.b_e = torch.from_numpy(self.w[f"{p}.joint.enc.bias"]).cuda()

    @staticmethod
    def get(case):
        key = (case["shape"], case["quant"])
        if key not in _models:
            _models[key] = _Model(*key)
        return _models[key]


# ---------------------------------------------------------------- inputs

def _lengths(case, seed):
    n, hi = case["sessions"], case["frames"]
    lo = case.get("frames_lo", hi)
    body = np.random.default_rng([seed, 1]).integers(lo, hi + 1, size=n) if lo < hi else np.full(n, hi)
    return body.astype(np.int32)


def _script(case, rows, rng):
    """Token and duration each frame speaks for (-1: blank)."""
    kind = synth.SHAPES[case["shape"]]["kind"]
    vocab = synth.SHAPES[case["shape"]]["vocab"]
    # talk and silence alternate; runs of about 25 frames on average
    flips = rng.random(rows) < 1 / 25
    level = rng.random(rows)
    run = np.cumsum(flips)
    talk = level[np.maximum.accumulate(np.where(flips, np.arange(rows), 0))] < case["speech"]
    p_tok = np.where(talk, 0.6 if kind == "tdt" else 0.3, 0.03)
    tok = rng.integers(1, min(vocab, 1025), size=rows) if kind == "eou" else rng.integers(1, vocab, size=rows)
    says = rng.random(rows) < p_tok
    y = np.where(says, tok, -1)
    if kind == "eou":   # the end of a turn, at some of the pauses
        y = np.where(flips & ~talk & (rng.random(rows) < 0.7), synth.SHAPES["eou-120m"]["eou_id"], y)
        return y, np.zeros(rows, np.int64)
    u = rng.random(rows)
    d = np.where(says, np.searchsorted(np.cumsum(TOKEN_DURATIONS), u), np.searchsorted(np.cumsum(BLANK_DURATIONS), u))
    return y, np.minimum(d, 4)


def _frames(case, seed, m, rows):
    """[rows, D] encoder frames on the GPU."""
    y, d = _script(case, rows, np.random.default_rng([seed, 2]))
    y, d = torch.from_numpy(y).cuda(), torch.from_numpy(d).cuda()
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = torch.empty(rows, m.info.D, device="cuda")
    blank, V1 = m.info.blank, m.info.V1
    for a in range(0, rows, CHUNK):
        yy, dd = y[a:a + CHUNK], d[a:a + CHUNK]
        says = (yy >= 0).unsqueeze(1)
        e = torch.where(says, A_TOK * m.z[yy.clamp(min=0)] + A_AFTER * m.z[blank], A_BLANK * m.z[blank].unsqueeze(0))
        if m.info.Dn:
            e = e + A_DUR * m.z[V1 + dd]
        f = (e - m.b_e) @ m.pinv
        out[a:a + CHUNK] = f + 0.1 * torch.randn(f.shape, generator=g, device="cuda")
    return out


def _inputs(case, seed):
    m = _Model.get(case)
    T = _lengths(case, seed)
    per = T * case["calls"] + TAIL                  # frames of a session
    rows = int(per.sum())
    enc = _frames(case, seed, m, rows)
    first = np.concatenate([[0], np.cumsum(per)[:-1]]).astype(np.int64)
    # the windows of each call: first row and length per session
    calls = [(first + c * T.astype(np.int64), T) for c in range(case["calls"])]
    calls.append((first + case["calls"] * T.astype(np.int64), np.full(len(T), TAIL, np.int32)))
    off = None
    if case["offsets"]:
        off = np.random.default_rng([seed, 3]).choice(np.array([0.0, 2.0, 4.0], np.float32), size=len(T))
    return m, enc, calls, off


def _caps(case):
    """Token capacity per session of each window."""
    return [2 * case["frames"] + 16] * case["calls"] + [2 * TAIL + 16]


def prepare(case, seed):
    m, enc, calls, off = _inputs(case, seed)
    n, info = case["sessions"], m.info
    state = dict(case=case, m=m, off=off, calls=calls, reset=np.ones(n, np.uint8))
    if case["host"]:
        host = enc.cpu().numpy()
        state["enc"] = [[host[r:r + t] for r, t in zip(rows, T)] for rows, T in calls]
        return state
    caps = _caps(case)
    state["enc"] = enc
    state["slots"] = np.arange(n, dtype=np.int32)
    state["outs"] = [dict(tokens=torch.zeros(n, c, dtype=torch.int32, device="cuda"),
                          n_tokens=torch.zeros(n, dtype=torch.int32, device="cuda"),
                          steps=torch.zeros(n, dtype=torch.int32, device="cuda"),
                          ctrl=torch.zeros(n, pk.PK_CTRL_N, dtype=torch.int32, device="cuda"),
                          segments=torch.zeros(n, c, dtype=torch.int32, device="cuda"),
                          n_segments=torch.zeros(n, dtype=torch.int32, device="cuda")) for c in caps]
    state["logits"] = torch.zeros(n, info.Vo, device="cuda")
    # the call descriptors, as a C program fills them once per buffer set
    state["batches"] = []
    for i, ((rows, T), o) in enumerate(zip(calls, state["outs"])):
        b = pk.PkBatch()
        b.n_utts, b.mem, b.d_enc, b.max_symbols = n, pk.MEM_DEVICE, info.D, info.max_symbols
        b.enc, b.enc_row, b.n_frames = enc.data_ptr(), rows.ctypes.data, T.ctypes.data
        b.slot = state["slots"].ctypes.data
        b.blank_bias = off.ctypes.data if off is not None else None
        b.tokens, b.token_cap = o["tokens"].data_ptr(), o["tokens"].shape[1]
        b.n_tokens, b.steps, b.ctrl_out = o["n_tokens"].data_ptr(), o["steps"].data_ptr(), o["ctrl"].data_ptr()
        if info.kind == pk.KIND_EOU:
            b.segments, b.seg_cap = o["segments"].data_ptr(), o["segments"].shape[1]
            b.n_segments = o["n_segments"].data_ptr()
        if i == 0:
            b.reset = state["reset"].ctypes.data
        if i == len(calls) - 1:
            b.logits, b.logit_steps = state["logits"].data_ptr(), 1
        state["batches"].append(b)
    torch.cuda.synchronize()
    return state


def run(state):
    m = state["m"]
    if not state["case"]["host"]:
        for b in state["batches"]:
            pk.check(pk.lib().pk_decode(m.dec.h, b))
        return _answer(state, state["outs"], state["logits"])
    got, logits = [], None
    last = len(state["enc"]) - 1
    for i, enc in enumerate(state["enc"]):
        r = m.dec.decode(enc, blank_bias=state["off"], reset=state["reset"] if i == 0 else None,
                         logit_steps=1 if i == last else 0)
        cap = _caps(state["case"])[i]
        o = dict(tokens=np.zeros((len(r), cap), np.int32), n_tokens=np.zeros(len(r), np.int32),
                 steps=np.zeros(len(r), np.int32), ctrl=np.zeros((len(r), pk.PK_CTRL_N), np.int32),
                 segments=np.zeros((len(r), cap), np.int32), n_segments=np.zeros(len(r), np.int32))
        for u, x in enumerate(r):
            o["tokens"][u, :len(x["tokens"])] = x["tokens"]
            o["segments"][u, :len(x["segments"])] = x["segments"]
            o["n_tokens"][u], o["steps"][u], o["n_segments"][u] = len(x["tokens"]), x["steps"], len(x["segments"])
            o["ctrl"][u] = x["ctrl"]
        got.append(o)
        if i == last:
            logits = np.stack([x["logits"][0] for x in r])
    return _answer(state, got, logits)


def _answer(state, outs, logits):
    got = dict(windows=_collect(outs), logits=logits)
    if state["case"]["sessions"] == 1:      # a single session is parked: its LSTM state comes back too
        s = state["m"].dec.read_state(0)
        got["h"], got["c"] = s["h"], s["c"]
    return got


def _collect(outs):
    """Each array of the equal windows as one (their sizes agree), the last window's apart."""
    stack = torch.stack if isinstance(outs[0]["steps"], torch.Tensor) else np.stack
    return dict(body={k: stack([o[k] for o in outs[:-1]]) for k in outs[0]}, tail=outs[-1])


# ---------------------------------------------------------------- work and tolerance

def _expected(case):
    """Steps and tokens of a pass, by the decode rules over a script of its kind."""
    kind = synth.SHAPES[case["shape"]]["kind"]
    T = _lengths(case, 0)
    frames = int((T * case["calls"] + TAIL).sum())
    rows = min(frames, 20000)
    y, d = _script(case, rows, np.random.default_rng([0, 2]))
    steps = tokens = t = 0
    while t < rows:
        steps += 1
        tok = y[t] >= 0
        tokens += int(tok)
        if kind == "eou":
            steps += int(tok)                        # the blank that ends the frame
            t += 1
        elif d[t] == 0:
            steps += 1
            t += 1
        else:
            t += int(d[t])
    return frames, steps * frames / rows, tokens * frames / rows


def work(case):
    cfg = synth.SHAPES[case["shape"]]
    H, J, D, L, V1 = cfg["H"], cfg["J"], cfg["D"], cfg["L"], cfg["vocab"] + 1
    Vo = V1 + len(cfg.get("durations", []))
    frames, steps, tokens = _expected(case)
    per = {"q8_0": 34 / 32, "q5_0": 22 / 32, "q4_0": 18 / 32, "f16": 2.0, "f32": 4.0}[case["quant"]]
    weights = per * (8 * L * H * H + J * (H + D + Vo)) + 4 * (8 * L * H + 2 * J + Vo)
    rows = per * H * min(tokens, V1)                                     # embedding rows
    state = 2 * case["sessions"] * (case["calls"] + 1) * 2 * L * H * 4   # h and c, in and out of each call
    out = 4 * tokens + case["sessions"] * (Vo + 10 * (case["calls"] + 1)) * 4
    flops = 2.0 * frames * D * J + steps * 2.0 * J * Vo + tokens * (16.0 * L * H * H + 2.0 * H * J)
    return {"bytes": weights + rows + frames * D * 4.0 + state + out, "flops": flops}


def tolerance(case):
    # logits: 32-bit sums of exact products (measured 2e-7 to 6e-7 against 64 bits and between sum
    # orders).  Decisions are clear, so tokens, steps and state words agree; a share of 2e-4 leaves room
    # for a tie.
    return {"rel": 4e-6, "max": 4e-5, "differ": 2e-4}


# ---------------------------------------------------------------- the same decode in 64 bits

def exact(case, seed):
    m, enc, calls, off = _inputs(case, seed)
    cfg, info, p = m.cfg, m.info, m.prefix
    n, H, L = case["sessions"], cfg["H"], cfg["L"]
    w = {k: torch.from_numpy(v).cuda().double() for k, v in m.w.items()}
    bias = torch.zeros(n, dtype=torch.float64, device="cuda")
    if off is not None:
        bias = torch.from_numpy(off).cuda().double()
    emb = w[f"{p}.predict.embed.weight"]

    def lstm(tok, h, c):
        x = emb[tok]
        hs, cs = [], []
        for l in range(L):
            q = f"{p}.predict.lstm.{l}."
            g = x @ w[q + "w_ih"].T + w[q + "b_ih"] + h[l] @ w[q + "w_hh"].T + w[q + "b_hh"]
            i, f, a, o = g.split(H, 1)
            cl = torch.sigmoid(f) * c[l] + torch.sigmoid(i) * torch.tanh(a)
            x = torch.sigmoid(o) * torch.tanh(cl)
            hs.append(x)
            cs.append(cl)
        return torch.stack(hs), torch.stack(cs)

    h = torch.zeros(L, n, H, dtype=torch.float64, device="cuda")
    c = torch.zeros_like(h)
    start = torch.full((n,), info.blank, device="cuda")
    h, c = lstm(start, h, c)
    h0, c0 = h[:, :1].clone(), c[:, :1].clone()      # a fresh state, and one after an end of turn
    sym = torch.zeros(n, dtype=torch.int64, device="cuda")
    carry = torch.zeros_like(sym)
    logits = torch.zeros(n, info.Vo, dtype=torch.float64, device="cuda")
    special = torch.from_numpy(np.resize(info.special, info.V1)).cuda().bool()
    special[len(info.special):] = False
    w_p, b_p = w[f"{p}.joint.pred.weight"], w[f"{p}.joint.pred.bias"]
    w_e, b_e = w[f"{p}.joint.enc.weight"], w[f"{p}.joint.enc.bias"]
    w_o, b_o = w[f"{p}.joint.out.weight"], w[f"{p}.joint.out.bias"]
    for k, (rows, T) in enumerate(calls):
        first, T = torch.from_numpy(rows).cuda(), torch.from_numpy(T).cuda().long()
        t = torch.minimum(carry, T)
        if info.kind == pk.KIND_EOU:
            sym = torch.where(T > 0, 0, sym)
        new = torch.ones(n, dtype=torch.bool, device="cuda")   # the window's first step is to come
        while bool((t < T).any()):
            u = torch.nonzero(t < T).squeeze(1)
            x = enc[first[u] + t[u]].double() @ w_e.T + b_e + h[L - 1, u] @ w_p.T + b_p
            z = torch.relu(x) @ w_o.T + b_o
            z[:, info.blank] += bias[u]
            if k == len(calls) - 1:
                at = new[u]
                logits[u[at]] = z[at]
                new[u] = False
            tok = z[:, :info.V1].argmax(1)
            if info.kind == pk.KIND_TDT:
                dur = z[:, info.V1:].argmax(1)
                adv = dur.clamp(min=1)
                say = tok != info.blank
                sym[u] = torch.where(say, sym[u] + 1, 0)
                move = ~say | (dur > 0) | (sym[u] >= info.max_symbols)
                t[u] += torch.where(move, adv, 0)
                sym[u] = torch.where(move, 0, sym[u])
                turn = torch.zeros_like(say)
            else:
                turn = tok == info.eou_id
                say = ~(turn | (tok == info.blank) | (tok == info.eob_id) | special[tok])
                sym[u] = torch.where(say, sym[u] + 1, sym[u])
                move = ~say | (sym[u] >= info.max_symbols)
                t[u] += move.long()
                sym[u] = torch.where(move & (t[u] < T[u]), 0, sym[u])
            if bool(say.any()):
                v = u[say]
                h[:, v], c[:, v] = lstm(tok[say], h[:, v], c[:, v])
            if bool(turn.any()):
                v = u[turn]
                h[:, v], c[:, v] = h0.expand(-1, len(v), -1), c0.expand(-1, len(v), -1)
        carry = (t - T).clamp(min=0)
    got = dict(windows=None, logits=logits)
    if n == 1:
        got["h"], got["c"] = h[:, 0].reshape(-1), c[:, 0].reshape(-1)
    return got
