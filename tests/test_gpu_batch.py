"""Decode batches of 5 to 16 sequences against the same sequences one at a time:
the rows' GEMVs, the chunk attention whose merge is a launch of its own or part of
the O projection's quantization, and batches of up to four with many chunks.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"\n[case] {msg}", flush=True)


LENS = [1, 31, 32, 33, 200, 511, 512, 513, 640, 700, 5, 64, 300, 90, 17, 400]


@pytest.mark.parametrize("lens", [LENS[:5], LENS[4:10], LENS[7:16], LENS,
                                  [900, 1000, 960, 1010]], ids=["5", "6", "9", "16", "long4"])
def test_batch_equals_single(gpu, lens):
    """Logits of two steps (the second feeds what the first appended) within 1e-5
    (2-norm) of each sequence decoded alone: both are within about 2e-6 of 64 bits
    on six layers."""
    ms = gpu
    say(f"batch of {len(lens)} against single sequences")
    arch = ms.arch_e4b(max_full_seq=1024, n_layers=6, vocab=4096)
    B, V = len(lens), 4096
    rng = np.random.default_rng(B)
    prompts = [rng.integers(0, V, n).tolist() for n in lens]
    nxt = rng.integers(0, V, B).tolist()

    def steps(model, seqs, tok, pos):
        tap = ms.DeviceBuffer(len(seqs) * V * 4)
        model.set_taps(None, tap)
        out = []
        for s in range(2):
            model.decode(tok, [p + s for p in pos], 1)
            out.append(tap.download(np.float32, (len(seqs), V)))
        model.set_taps(None, None)
        return out

    m = ms.Model(arch, max_seqs=B, max_rows=1, max_pos=1030)
    m.fill_synthetic(42)
    for b, p in enumerate(prompts):
        m.prefill(p, 0, b)
    got = steps(m, prompts, nxt, lens)
    m.close()
    one = ms.Model(arch, max_seqs=1, max_rows=1, max_pos=1030)
    one.fill_synthetic(42)
    for b, p in enumerate(prompts):
        one.reset()
        one.prefill(p, 0, 0)
        ref = steps(one, [p], [nxt[b]], [lens[b]])
        for s in range(2):
            d = np.linalg.norm(got[s][b] - ref[s][0]) / np.linalg.norm(ref[s][0])
            assert d < 1e-5, (b, s, d)
    one.close()


@pytest.mark.parametrize("lens", [[1], [700], LENS[:3], LENS[4:8], LENS[5:10], LENS],
                         ids=["first", "1", "3", "4", "5", "16"])
def test_14b_batch_equals_prefill(gpu, lens):
    """Five query heads of 128 per kv head: logits of a decode step within 1e-5 of
    those that a prefill of the prompt and its next token gives (the flash
    attention and the GEMM: other kernels throughout)."""
    ms = gpu
    say(f"14B class, batch of {len(lens)} against prefill")
    V = 4096
    arch = ms.arch_14b(max_len=1024, n_layers=2, vocab=V)
    B = len(lens)
    rng = np.random.default_rng(100 + B)
    prompts = [rng.integers(0, V, n).tolist() for n in lens]
    nxt = rng.integers(0, V, B).tolist()
    m = ms.Model(arch, max_seqs=B, max_rows=1, max_pos=1024)
    m.fill_synthetic(42)
    for b, p in enumerate(prompts):
        m.prefill(p, 0, b)
    tap = ms.DeviceBuffer(B * V * 4)
    m.set_taps(None, tap)
    m.decode(nxt, list(lens), 1)
    got = tap.download(np.float32, (B, V))
    m.set_taps(None, None)
    m.close()
    one = ms.Model(arch, max_seqs=1, max_rows=1, max_pos=1024)
    one.fill_synthetic(42)
    tap1 = ms.DeviceBuffer(V * 4)
    one.set_taps(None, tap1)
    for b, p in enumerate(prompts):
        one.reset()
        one.prefill(p + [nxt[b]], 0, 0)
        ref = tap1.download(np.float32, V)
        d = np.linalg.norm(got[b] - ref) / np.linalg.norm(ref)
        assert d < 1e-5, (b, d)
    one.close()


@pytest.mark.parametrize("kind,B", [("14b", 1), ("14b", 6), ("e4b", 1), ("e4b", 3), ("e4b", 6)])
def test_attention_sweep_of_each_decode_path(gpu, kind, B):
    """ms_prof_sweep re-runs the attention launch of the profiled step, whichever path the
    step takes: on every layer of its kind, with the K and V rows of every attended key as
    bytes, and without a trace in what the model decodes next."""
    ms = gpu
    say(f"attention sweep {kind} B={B}")
    V, n = 4096, 90
    arch = (ms.arch_14b(max_len=256, n_layers=3, vocab=V) if kind == "14b"
            else ms.arch_e4b(max_full_seq=256, n_layers=6, vocab=V))
    m = ms.Model(arch, max_seqs=B, max_rows=1, max_pos=256)
    m.fill_synthetic(42)
    rng = np.random.default_rng(B)
    prompts = [rng.integers(0, V, n + b).tolist() for b in range(B)]
    nxt = rng.integers(0, V, B).tolist()

    def run(sweep):
        m.reset()
        for b, p in enumerate(prompts):
            m.prefill(p, 0, b)
        ms.prof_enable(sweep)
        ids = [m.decode(nxt, [len(p) for p in prompts], 2, use_graph=False)]
        ms.prof_enable(False)
        if sweep:
            sw = ms.prof_sweep(m, "attention", passes=2)
            # (the E4B's sliding layers, five of six)
            layers = [d for d in arch.layers if kind == "14b" or d.cache_kind == 1]
            d = layers[0]
            # (positions after the two steps)
            keys = sum(min(len(p) + 3, d.cache_len) for p in prompts)
            assert sw["launches"] == 2 * len(layers) and sw["avg_us"] > 0
            assert sw["bytes_per_launch"] == 2.0 * keys * d.kv_dim * 4
        ids.append(m.decode_continue(3, B, use_graph=False))
        return np.concatenate(ids)

    a, b = run(False), run(True)
    m.close()
    assert np.array_equal(a, b)
    with pytest.raises(Exception):
        other = ms.Model(arch, max_seqs=1, max_rows=1, max_pos=256)
        try:
            ms.prof_sweep(other, "attention")  # nothing recorded: its launches are gone
        finally:
            other.close()


# heads, kv heads, head dim, length of a circular cache (0: linear): one to three and six to eight query
# heads per kv head, the most heads and the longest rows of the merge in O's quantization
SHAPES = [(2, 2, 128, 0), (4, 2, 128, 64), (6, 2, 128, 0), (12, 2, 128, 50), (14, 2, 128, 0),
          (16, 2, 128, 0), (48, 8, 128, 100), (2, 2, 256, 0), (2, 1, 256, 64), (3, 1, 256, 0),
          (1, 1, 512, 0), (2, 1, 512, 0), (3, 1, 512, 77), (16, 4, 512, 0)]


@pytest.mark.parametrize("B", [1, 3, 6, 16])
@pytest.mark.parametrize("nh,nkv,hd,circ", SHAPES)
def test_decode_attention_shapes(gpu, nh, nkv, hd, circ, B):
    """One layer, row by row, against the float64 statement of it: sequences at positions
    of their own, 0 to past 128 (below 64 one launch, past it chunks and their merge; with
    five rows or more the merge is in O's quantization).  Q4 rows carry 31 bits, everything
    else is fp32: a row is within 2e-6 of 64 bits, as the other layers' tests hold it."""
    from tests.golden.layer_ref import RefLayer
    ms = gpu
    say(f"decode attention nh={nh} nkv={nkv} hd={hd} circular={circ} B={B}")
    D, n = 256, 133
    desc = ms.LayerDesc(q_dim=nh * hd, kv_dim=nkv * hd, head_dim=hd, n_heads=nh, n_kv_heads=nkv,
                        rot_dim=hd // 2, theta=1e4, cache_kind=int(circ > 0),
                        cache_len=circ or 141, clamp_reads=0)
    arch = ms.Arch("one", D, D, [desc])
    rng = np.random.default_rng(nh * hd + B)
    w = [rng.integers(1, 16, (k, c // 2 * 2)).astype(np.uint8) for k, c in arch.matrix_shapes(0)]
    w = [(a[:, 0::2] | (a[:, 1::2] << 4)).astype(np.uint8) for a in w]
    sc = [np.float32(1 / (4.3 * np.sqrt(k))) for k, _ in arch.matrix_shapes(0)]
    m = ms.Model(arch, max_seqs=B, max_rows=1, max_pos=160)
    for i in range(7):
        m.set_matrix(0, i, w[i], float(sc[i]))
    m.set_ple(0, 1.0)
    x = rng.standard_normal((B, n, D)).astype(np.float32)
    lag = [5 * b % 31 for b in range(B)]
    got = np.zeros((B, n, D), np.float32)
    for t in range(n):
        # (a sequence that lags repeats its first row, which writes the same keys)
        pos = [max(0, t - s) for s in lag]
        out = m.layer_forward(0, np.stack([x[b, p] for b, p in enumerate(pos)]), pos, 1)
        for b, p in enumerate(pos):
            got[b, p] = out[b]
    m.close()
    for b in {0, B // 2, B - 1}:
        k = n - lag[b]
        ref = RefLayer(desc, D, D, w, sc, 1.0).forward(x[b, :k].astype(np.float64), 0)
        err = np.linalg.norm(got[b, :k] - ref, axis=1) / np.linalg.norm(ref, axis=1)
        assert err.max() < 2e-6, (b, int(err.argmax()), err.max())
