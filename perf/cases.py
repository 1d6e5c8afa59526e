"""The calls whose speed matters to a user of this framework, with sizes from
its own architectures (E4B, 14B class, demo), tests and benchmark.

A case is one pass through public entry points: a Q4 product, a forward step of
the demo harness, greedy decode steps, a prompt's prefill, the head with a
sampled draw, or the converter's quantization of one weight.  Inputs come from
torch generators seeded per case; `exact` restates each computation in 64 bits.
"""
import ctypes
import math

import numpy as np
import torch

import mojostream_amd as ms

# ---- the cases ---------------------------------------------------------------


def listed():
    return [
        # the smallest call: one row times a small square matrix (the Q4
        # benchmark's first shape); launch latency sets it
        {"name": "q4_1x1024x1024", "kind": "q4", "M": 1, "K": 1024, "N": 1024},
        # a ragged handful of rows on the E4B FFN shape: a batch of 13
        # sequences or the tail of a prompt
        {"name": "q4_13x2560x10240", "kind": "q4", "M": 13, "K": 2560, "N": 10240},
        # the Q4 benchmark's largest shape
        {"name": "q4_64x4096x4096", "kind": "q4", "M": 64, "K": 4096, "N": 4096},
        # one step of the harness loop: four fresh rows through the demo model
        {"name": "forward_demo_4rows", "kind": "forward", "arch": "demo", "rows": 4, "base": 200},
        # interactive generation: one sequence, a short prompt behind it
        {"name": "decode_e4b_b1", "kind": "decode", "arch": "e4b", "seqs": 1, "ctx": 128, "steps": 4},
        # four users at once
        {"name": "decode_e4b_b4", "kind": "decode", "arch": "e4b", "seqs": 4, "ctx": 300, "steps": 4},
        # the largest batch a model takes, past the sliding window
        {"name": "decode_e4b_b16", "kind": "decode", "arch": "e4b", "seqs": 16, "ctx": 640, "steps": 1},
        # a chat turn: time to the first token of a short prompt
        {"name": "prefill_e4b_77", "kind": "prefill", "arch": "e4b", "tokens": 77},
        # a long prompt: the time to first token of the benchmark
        {"name": "prefill_e4b_2048", "kind": "prefill", "arch": "e4b", "tokens": 2048},
        # layers of the 14B class (five query heads per kv head), a document
        {"name": "prefill_14b_1000", "kind": "prefill", "arch": "14b", "tokens": 1000},
        # one token of sampled generation: head, repetition penalty, draw
        {"name": "sample_262144", "kind": "sample", "head": "q4", "D": 2560, "vocab": 262144,
         "temperature": 0.8, "penalty": 1.2, "history": 600},
        # the converter on one FFN weight of a checkpoint
        {"name": "quantize_bf16_10240x2560", "kind": "quantize", "dtype": "BF16",
         "n_out": 10240, "n_in": 2560},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("q4", "q4", "forward", "decode", "decode", "prefill", "prefill",
                       "sample", "quantize"))
    if kind == "q4":
        return {"kind": kind, "M": _log(rng, 1, 512), "K": 128 * _log(rng, 4, 80),
                "N": 16 * _log(rng, 32, 1024)}
    if kind == "forward":
        return {"kind": kind, "arch": "demo", "rows": rng.randint(1, 4),
                "base": rng.randint(0, 400)}
    if kind == "decode":
        arch = rng.choice(("e4b", "e4b", "14b"))
        seqs = _log(rng, 1, 16)
        ctx = _log(rng, 16, 1500 if seqs <= 4 else 700)
        # past the window one step a pass, so that a repeated pass sees the same cache
        return {"kind": kind, "arch": arch, "seqs": seqs, "ctx": ctx,
                "steps": rng.randint(1, 4) if ctx + 4 <= 512 else 1}
    if kind == "prefill":
        arch = rng.choice(("e4b", "e4b", "14b"))
        return {"kind": kind, "arch": arch, "tokens": _log(rng, 17, 2048)}
    if kind == "sample":
        return {"kind": kind, "head": rng.choice(("q4", "q4", "f32")),
                "D": rng.choice((1024, 2560, 5120)), "vocab": 64 * _log(rng, 500, 4096),
                "temperature": rng.choice((0.0, round(rng.uniform(0.3, 1.0), 2))),
                "penalty": rng.choice((1.0, round(rng.uniform(1.05, 1.3), 2))),
                "history": _log(rng, 1, 4000)}
    return {"kind": "quantize", "dtype": rng.choice(("BF16", "BF16", "F16", "F32")),
            "n_out": 2 * _log(rng, 256, 6900), "n_in": _log(rng, 512, 10240)}


# ---- architectures -------------------------------------------------------------

# layers and head size of the models the cases run; the 14B class with four of
# its 48 layers, all alike
_MAX_POS = 2560


def _arch(name):
    if name == "demo":
        return ms.arch_demo(max_len=512)
    if name == "14b":
        return ms.arch_14b(max_len=_MAX_POS, n_layers=4)
    return ms.arch_e4b(max_full_seq=_MAX_POS)


def _gen(*key):
    s = 0x9E3779B97F4A7C15
    for k in key:
        s = ((s ^ (int(k) + 0x632BE59BD9B4E019)) * 0xBF58476D1CE4E5B9) & ((1 << 63) - 1)
        s ^= s >> 29
    g = torch.Generator(device="cuda")
    g.manual_seed(s)
    return g


def _q4_bytes(K, N, *key):
    """Row-major Q4 bytes [K][N/2] of a zero-mean weight (nibbles 1..15)."""
    b = torch.randint(0, 256, (K, N // 2), dtype=torch.uint8, device="cuda", generator=_gen(*key))
    b |= ((b & 15) == 0).to(torch.uint8) * 8
    b |= ((b >> 4) == 0).to(torch.uint8) * 128
    return b


def _scale(K, gain, u):
    return float(np.float32(gain * u / (ms.BALANCED_NIBBLE_STD * math.sqrt(K))))


class _Weights:
    """The seeded weights of a model, made one matrix at a time."""

    def __init__(self, arch, seed):
        self.arch, self.seed = arch, seed
        r = np.random.RandomState(seed % (1 << 31))
        self.u = r.uniform(0.8, 1.2, (arch.n_layers, 7))
        self.ple = [float(np.float32(v)) for v in r.uniform(0.8, 1.2, arch.n_layers)]
        self.gamma = r.uniform(0.8, 1.2, arch.hidden).astype(np.float32)

    def matrix(self, l, i):
        K, N = self.arch.matrix_shapes(l)[i]
        return _q4_bytes(K, N, self.seed, l, i), _scale(K, ms.BALANCED_GAINS[i], self.u[l, i])

    def head(self):
        D = self.arch.hidden
        return _q4_bytes(D, self.arch.vocab, self.seed, 1 << 20, 0), _scale(D, 1.0, 1.0)


class _Rows:
    """A torch tensor as the device buffer the model's taps take."""

    def __init__(self, *shape):
        self.t = torch.zeros(shape, dtype=torch.float32, device="cuda")
        self.ptr = self.t.data_ptr()


def _model(arch, seed, seqs, rows):
    w = _Weights(arch, seed)
    m = ms.Model(arch, max_seqs=seqs, max_rows=rows,
                 max_pos=512 if arch.vocab == 0 else _MAX_POS)
    for l in range(arch.n_layers):
        keep = [w.matrix(l, i) for i in range(7)]
        torch.cuda.synchronize()
        for i, (b, s) in enumerate(keep):
            m.set_matrix_device(l, i, b.data_ptr(), s)
        m.set_ple(l, w.ple[l])
        ms.synchronize()
    if arch.vocab:
        b, s = w.head()
        torch.cuda.synchronize()
        m.set_lm_head(None, s, gamma=w.gamma, dptr=b.data_ptr())
        ms.synchronize()
    return m


def _tokens(n, vocab, *key):
    g = torch.Generator()
    g.manual_seed(_gen(*key).initial_seed())
    return torch.randint(0, vocab, (n,), generator=g).tolist()


def _decode_inputs(case, vocab, seed):
    """Prompt and next token of every sequence; the lengths of a batch differ."""
    B, ctx = case["seqs"], case["ctx"]
    lens = [max(1, ctx - (7 * b) % max(1, ctx // 4)) for b in range(B)]
    return [_tokens(n, vocab, seed, 77, b) for b, n in enumerate(lens)], \
        _tokens(B, vocab, seed, 78)


def _forward_rows(case, D, seed):
    n = case["base"] + case["rows"]
    return torch.randn((n, D), dtype=torch.float32, device="cuda", generator=_gen(seed, 5))


# ---- prepare and run -------------------------------------------------------------

_DT = {"F32": torch.float32, "BF16": torch.bfloat16, "F16": torch.float16}


def _q4_inputs(case, seed):
    M, K, N = case["M"], case["K"], case["N"]
    a = torch.randn((M, K), dtype=torch.float32, device="cuda", generator=_gen(seed, 1))
    return a, _q4_bytes(K, N, seed, 2), _scale(K, 1.0, 1.0)


def _sample_inputs(case, seed):
    D, V = case["D"], case["vocab"]
    x = torch.randn((1, D), dtype=torch.float32, device="cuda", generator=_gen(seed, 1))
    hist = torch.randint(0, V, (case["history"],), dtype=torch.int32, device="cuda",
                         generator=_gen(seed, 3))
    # generated text repeats itself
    hist[case["history"] // 2:] = hist[: case["history"] - case["history"] // 2].clone()
    # logits of standard deviation 3, as a head gives: a few likely tokens
    if case["head"] == "q4":
        return x, hist, _q4_bytes(D, V, seed, 2), _scale(D, 3.0, 1.0)
    w = torch.randn((D, V), dtype=torch.float32, device="cuda", generator=_gen(seed, 2))
    return x, hist, w.mul_(3.0 / math.sqrt(D)), 1.0


def _quantize_input(case, seed):
    w = torch.randn((case["n_out"], case["n_in"]), dtype=torch.float32, device="cuda",
                    generator=_gen(seed, 1))
    return (w * 0.02).to(_DT[case["dtype"]])


def prepare(case, seed):
    ms.init(0)
    kind = case["kind"]
    st = {"case": case, "seed": seed}
    if kind == "q4":
        M, K, N = case["M"], case["K"], case["N"]
        a, b, s = _q4_inputs(case, seed)
        w = torch.empty(K * N // 2, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        ms.check(ms.lib().ms_q4_pack(w.data_ptr(), b.data_ptr(), K, N))
        ms.synchronize()
        st.update(a=a, w=w, scale=s, c=torch.zeros((M, N), dtype=torch.float32, device="cuda"))
    elif kind == "sample":
        D, V = case["D"], case["vocab"]
        x, hist, w, s = _sample_inputs(case, seed)
        if case["head"] == "q4":
            p = torch.empty(D * V // 2, dtype=torch.uint8, device="cuda")
            torch.cuda.synchronize()
            ms.check(ms.lib().ms_q4_pack(p.data_ptr(), w.data_ptr(), D, V))
            ms.synchronize()
            w = p
        st.update(x=x, hist=hist, w=w, scale=s, logits=_Rows(1, V),
                  ids=torch.zeros(1, dtype=torch.int32, device="cuda"))
    elif kind == "quantize":
        w = _quantize_input(case, seed)
        st.update(w=w, q=torch.zeros((case["n_in"], case["n_out"] // 2), dtype=torch.uint8,
                                     device="cuda"))
    else:
        arch = _arch(case["arch"])
        if kind == "forward":
            T, base = case["rows"], case["base"]
            m = _model(arch, seed, 1, 4)
            x = _forward_rows(case, arch.hidden, seed)
            buf = torch.zeros((4, arch.hidden), dtype=torch.float32, device="cuda")
            torch.cuda.synchronize()
            for p in range(0, base, 4):  # the steps before this one fill the caches
                n = min(4, base - p)
                _step(m, buf, x[p:p + n], n, p)
            st.update(m=m, x=x[base:].contiguous(), buf=buf[:T])
        elif kind == "decode":
            m = _model(arch, seed, case["seqs"], 1)
            prompts, nxt = _decode_inputs(case, arch.vocab, seed)
            for b, p in enumerate(prompts):
                m.prefill(p, 0, b)
            logits = _Rows(case["seqs"], arch.vocab)
            m.set_taps(None, logits)
            st.update(m=m, tok=nxt, pos=[len(p) for p in prompts], logits=logits)
        else:
            m = _model(arch, seed, 1, 1)
            logits = _Rows(1, arch.vocab)
            m.set_taps(None, logits)
            st.update(m=m, tok=_tokens(case["tokens"], arch.vocab, seed, 77), logits=logits)
    torch.cuda.synchronize()
    return st


def _step(m, buf, rows, T, base):
    ms.check(ms.lib().ms_memcpy_d2d(buf.data_ptr(), rows.data_ptr(), rows.numel() * 4))
    ms.check(ms.lib().ms_forward(m.h, buf.data_ptr(), 1, T, (ctypes.c_int * 1)(base), None))


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "q4":
        ms.check(ms.lib().ms_q4_matmul(st["c"].data_ptr(), st["a"].data_ptr(),
                                       st["w"].data_ptr(), case["M"], case["K"], case["N"],
                                       st["scale"], 0))
        return st["c"]
    if kind == "forward":
        _step(st["m"], st["buf"], st["x"], case["rows"], case["base"])
        return st["buf"]
    if kind == "decode":
        ids = st["m"].decode(st["tok"], st["pos"], case["steps"])
        return {"ids": ids, "logits": st["logits"].t}
    if kind == "prefill":
        first = st["m"].prefill(st["tok"], 0, 0)
        return {"id": first, "logits": st["logits"].t}
    if kind == "sample":
        lg, D, V = st["logits"], case["D"], case["vocab"]
        if case["head"] == "q4":
            ms.check(ms.lib().ms_lm_head_argmax(st["x"].data_ptr(), 1, D, st["w"].data_ptr(), V,
                                                st["scale"], lg.ptr, st["ids"].data_ptr()))
        else:
            ms.check(ms.lib().ms_matmul_f32(lg.ptr, st["x"].data_ptr(), st["w"].data_ptr(),
                                            1, D, V, 0))
        h = _Hist(st["hist"])
        i = ms.sample(lg, V, case["temperature"], h, case["history"], case["penalty"],
                      st["seed"])
        return {"id": i, "values": lg.t}
    s = _quantize(st["q"], st["w"], case)
    return {"bytes": st["q"], "scale": s}


class _Hist:
    def __init__(self, t):
        self.ptr = t.data_ptr()


def _quantize(q, w, case):
    s = ctypes.c_float()
    ms.check(ms.lib().ms_q4_quantize(q.data_ptr(), ctypes.byref(s), w.data_ptr(),
                                     ms.Q4_DTYPES[case["dtype"]], case["n_out"], case["n_in"],
                                     32))
    return float(s.value)


# ---- what a pass cannot do without ------------------------------------------------


def _keys(d, p):
    """Keys that the row at position p attends to."""
    return min(p + 1, d.cache_len)


def work(case):
    kind = case["kind"]
    if kind == "q4":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": K * N / 2 + 4.0 * M * (K + N), "flops": 2.0 * M * K * N}
    if kind == "sample":
        D, V = case["D"], case["vocab"]
        w = D * V / 2 if case["head"] == "q4" else 4.0 * D * V
        return {"bytes": w + 4.0 * V + 4.0 * case["history"], "flops": 2.0 * D * V}
    if kind == "quantize":
        n = case["n_out"] * case["n_in"]
        return {"bytes": n * ((4 if case["dtype"] == "F32" else 2) + 0.5), "flops": 2.0 * n}
    arch = _arch(case["arch"])
    wb = arch.weight_bytes()
    head = arch.hidden * arch.vocab / 2
    if kind == "decode":
        pos = [len(p) for p in _decode_lens(case)]
        kv = att = 0.0
        for s in range(case["steps"]):
            for p in pos:
                for d in arch.layers:
                    kv += 8.0 * _keys(d, p + s) * d.kv_dim
                    att += 4.0 * _keys(d, p + s) * d.q_dim
        return {"bytes": case["steps"] * (wb + head + 4.0 * case["seqs"] * arch.vocab) + kv,
                "flops": case["steps"] * case["seqs"] * 4.0 * (wb + head) + att}
    if kind == "prefill":
        T, base = case["tokens"], 0
    else:
        T, base = case["rows"], case["base"]
    kv = att = 0.0
    for d in arch.layers:
        kv += 8.0 * (min(base, d.cache_len) + T) * d.kv_dim
        att += sum(4.0 * _keys(d, p) * d.q_dim for p in range(base, base + T))
    rows = 8.0 * T * arch.hidden if kind == "forward" else 4.0 * arch.vocab
    return {"bytes": wb + head + kv + rows, "flops": 4.0 * wb * T + 4.0 * head + att}


def _decode_lens(case):
    B, ctx = case["seqs"], case["ctx"]
    return [range(max(1, ctx - (7 * b) % max(1, ctx // 4))) for b in range(B)]


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    # Q4 products: activations in 22 or 31 bit fixed point, fp32 results; 3.7e-7
    # from 64 bits
    if kind == "q4":
        return {"rel": 1.5e-6, "max": 1.5e-5}
    # probabilities of a softmax over fp32 logits, which are up to about 20 and
    # good to 1e-7 of that
    if kind == "sample":
        return {"rel": 1e-5, "max": 1e-4}
    # whole models in fp32: rounding grows through the layers; 1.8e-6 from 64 bits
    return {"rel": 8e-6, "max": 1e-4}


# ---- the same in 64 bits ------------------------------------------------------------


def _deq(b, scale):
    """Row-major Q4 bytes as float64 weights."""
    w = torch.empty((b.shape[0], 2 * b.shape[1]), dtype=torch.float64, device="cuda")
    w[:, 0::2] = (b & 15).double()
    w[:, 1::2] = (b >> 4).double()
    return w.sub_(8.0).mul_(scale)


def _rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)


def _rope(x, rot, theta):
    """x [n][heads][hd], row p at position p; angles in fp32, as the model
    defines them."""
    half, n = rot // 2, x.shape[0]
    i = np.arange(half, dtype=np.float32)
    f = np.exp(-(np.float32(2) * i) / np.float32(rot) * np.float32(math.log(theta)),
               dtype=np.float32)
    ang = np.arange(n, dtype=np.float32)[:, None] * f[None, :]
    a64 = torch.from_numpy(ang.astype(np.float64)).cuda()
    c, s = torch.cos(a64)[:, None, :], torch.sin(a64)[:, None, :]
    y = x.clone()
    a, b = x[..., :half], x[..., half:rot]
    y[..., :half] = a * c - b * s
    y[..., half:rot] = a * s + b * c
    return y


def _attend(d, q, k, v):
    """Causal attention of all rows; q [n][heads][hd], k and v [n][kv heads][hd]."""
    n = q.shape[0]
    out = torch.empty_like(q)
    p = torch.arange(n, device="cuda")
    for h in range(d.n_heads):
        kh = h // (d.n_heads // d.n_kv_heads)
        kk, vv = k[:, kh].contiguous(), v[:, kh].contiguous()
        for r0 in range(0, n, 1024):
            r1 = min(n, r0 + 1024)
            s = torch.matmul(q[r0:r1, h].contiguous(), kk.t().contiguous()) / math.sqrt(d.head_dim)
            ahead = p[None, :] - p[r0:r1, None]
            hide = ahead > 0
            if d.cache_kind == ms.MS_CACHE_CIRCULAR:
                hide |= ahead <= -d.cache_len
            s.masked_fill_(hide, -math.inf)
            out[r0:r1, h] = torch.matmul(torch.softmax(s, -1), vv)
    return out


def _exact_layers(arch, w, seqs):
    """Rows after the last layer; seqs: input rows of each sequence from position 0."""
    lens = [x.shape[0] for x in seqs]
    x = torch.cat(seqs)
    for l, d in enumerate(arch.layers):
        mat = lambda i: _deq(*w.matrix(l, i))  # noqa: E731
        x = _rms(x * w.ple[l])
        q = torch.matmul(x, mat(0)).view(-1, d.n_heads, d.head_dim)
        k = torch.matmul(x, mat(1)).view(-1, d.n_kv_heads, d.head_dim)
        v = torch.matmul(x, mat(2)).view(-1, d.n_kv_heads, d.head_dim)
        att, r = [], 0
        for n in lens:
            att.append(_attend(d, _rope(q[r:r + n], d.rot_dim, d.theta),
                               _rope(k[r:r + n], d.rot_dim, d.theta), v[r:r + n]))
            r += n
        x = _rms(x + torch.matmul(torch.cat(att).reshape(-1, d.q_dim), mat(3)))
        g = torch.matmul(x, mat(4))
        x = x + torch.matmul(torch.matmul(x, mat(5)) * g * torch.sigmoid(g), mat(6))
    return list(x.split(lens))


def _exact_head(arch, w, rows):
    b, s = w.head()
    y = _rms(rows) * torch.from_numpy(w.gamma.astype(np.float64)).cuda()
    return torch.cat([torch.matmul(y, _deq(b[:, c:c + 16384].contiguous(), s))
                      for c in range(0, b.shape[1], 16384)], 1)


def _embed(w, tokens):
    b, s = w.head()
    t = torch.tensor(tokens, device="cuda")
    col = b[:, t // 2]
    nib = torch.where(t % 2 == 1, col >> 4, col & 15)
    # the embedding row itself is an fp32 product
    return ((nib.float() - 8.0) * s).t().contiguous().double()


def _exact_sample(case, seed):
    x, hist, w, s = _sample_inputs(case, seed)
    V = case["vocab"]
    cols = [w[:, c:c + 16384] for c in range(0, w.shape[1], 16384)]
    v = torch.cat([torch.matmul(x.double(), _deq(c, s) if case["head"] == "q4" else c.double())
                   for c in cols], 1)
    v = v[0]
    if case["penalty"] > 1.0:
        pen = float(np.float32(case["penalty"]))
        n = torch.bincount(hist.long(), minlength=V).double()
        f = torch.pow(torch.full_like(n, pen), n)
        v = torch.where(v > 0, v / f, v * f)
    if case["temperature"] > 0.01:
        v = torch.softmax((v - v.max()) / float(np.float32(case["temperature"])), 0)
    return {"id": None, "values": v[None]}


def exact(case, seed):
    kind = case["kind"]
    if kind == "q4":
        a, b, s = _q4_inputs(case, seed)
        return torch.matmul(a.double(), _deq(b, s))
    if kind == "sample":
        return _exact_sample(case, seed)
    if kind == "quantize":
        w = _quantize_input(case, seed)
        return {"bytes": None, "scale": float(w.double().abs().max()) / 7.0}
    arch = _arch(case["arch"])
    w = _Weights(arch, seed)
    if kind == "forward":
        x = _forward_rows(case, arch.hidden, seed).double()
        return _exact_layers(arch, w, [x])[0][case["base"]:]
    if kind == "prefill":
        rows = _embed(w, _tokens(case["tokens"], arch.vocab, seed, 77))
        return {"id": None, "logits": _exact_head(arch, w, _exact_layers(arch, w, [rows])[0][-1:])}
    if case["seqs"] * case["ctx"] > 12000:
        # the longest batches take too long in 64 bits
        return None
    prompts, nxt = _decode_inputs(case, arch.vocab, seed)
    seqs = [p + [t] for p, t in zip(prompts, nxt)]
    while True:
        last = torch.cat([y[-1:] for y in
                          _exact_layers(arch, w, [_embed(w, q) for q in seqs])])
        logits = _exact_head(arch, w, last)
        if len(seqs[0]) == len(prompts[0]) + case["steps"]:
            return {"ids": None, "logits": logits}
        seqs = [q + [int(t)] for q, t in zip(seqs, logits.argmax(1).tolist())]
