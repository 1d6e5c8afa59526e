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
