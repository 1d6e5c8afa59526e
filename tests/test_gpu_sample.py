"""ms_sample over rows whose slices and blocks are cut at their edges.

A row is 1024 slices; a block owns whole slices, up to 2048 logits, or, where a
slice is longer, one slice in passes of 2048.  The sizes lie at and around
those limits.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"\n[case] {msg}", flush=True)


SIZES = [1, 2, 255, 256, 257, 1023, 1024, 1025, 2047, 2049, 8193, 65537, 300001,
         1024 * 2048, 1024 * 2048 + 1, 1024 * 2100 + 7]


def _history(rng, V, n):
    """n ids, the second half repeating the first, some outside the row, one
    many times."""
    h = rng.integers(0, V, n).astype(np.int32)
    h[n // 2:] = h[: n - n // 2]
    h[:: 7] = h[0]
    if n > 4:
        h[1], h[2] = V, -1
    return h


@pytest.mark.parametrize("V", SIZES)
def test_sample_edges_vs_oracle(gpu, oracle, V):
    """Greedy: id and penalized logits equal the oracle's bit for bit.  Draws:
    the probabilities within 2e-4 of 64 bits (sums of up to 2100 values in a
    slice, then of 1024 slices, each addition off by 2^-24 at most: 1.9e-4; the
    exponents' rounding adds 5e-6), the id where their 64-bit sum crosses the
    target, up to the same rounding."""
    ms = gpu
    say(f"sample edges V={V}")
    rng = np.random.default_rng(V)
    logits = (rng.standard_normal(V) * 3).astype(np.float32)
    logits[V // 2:: 97] = logits[V // 3]  # equal values: the first wins
    for n in (0, 5, 600, 8192):
        hist = _history(rng, V, n) if n else np.zeros(0, np.int32)
        dh = ms.DeviceBuffer.from_array(hist if n else np.zeros(1, np.int32))
        dl = ms.DeviceBuffer.from_array(logits)
        gid = ms.sample(dl, V, 0.0, dh, n, 1.3, 7)
        oid, olog = oracle.sample(logits, 0.0, hist, 1.3, 7)
        assert gid == oid
        assert np.array_equal(dl.download(np.float32, V), olog)
        for seed, T in ((n + 1, 0.7), (n + 2, 1.4)):
            dl.upload(logits)
            gid = ms.sample(dl, V, T, dh, n, 1.2, seed)
            _, pen = oracle.sample(logits, 0.0, hist, 1.2, seed)
            p = dl.download(np.float32, V)
            x = (pen.astype(np.float64) - pen.max()) / np.float32(T)
            e = np.exp(x)
            np.testing.assert_allclose(p, e / e.sum(), rtol=2e-4, atol=1e-30)
            cdf = np.cumsum(p.astype(np.float64))
            target = oracle.sample_target(seed)
            lo = cdf[gid - 1] if gid > 0 else 0.0
            assert lo <= target + 2e-4 and (cdf[gid] >= target - 2e-4 or gid == V - 1)
        dh.free()
        dl.free()


def test_sample_odd_values(gpu):
    """No logit above -inf, and NaN: the index stays inside the row; a NaN is
    passed over by the maximum unless it comes first."""
    ms = gpu
    say("sample: -inf and NaN rows")
    V = 5000
    dh = ms.DeviceBuffer.from_array(np.zeros(1, np.int32))
    v = np.full(V, -np.inf, np.float32)
    dl = ms.DeviceBuffer.from_array(v)
    assert ms.sample(dl, V, 0.0, dh, 0, 1.0, 1) == 0
    v[4321] = -1.0
    v[100] = np.nan
    dl.upload(v)
    assert ms.sample(dl, V, 0.0, dh, 0, 1.0, 1) == 4321
    v[0] = np.nan
    dl.upload(v)
    assert ms.sample(dl, V, 0.0, dh, 0, 1.0, 1) == 0
    dl.upload(v)
    assert ms.sample(dl, V, 0.7, dh, 0, 1.0, 1) == V - 1
    dl.free()
    dh.free()


@pytest.mark.parametrize("V", [3000, 262144])
def test_sample_flat_tail(gpu, oracle, V):
    """One id holds nearly all the mass in the middle of the row: draws on it, and
    draws whose target lies within rounding of many slices of next to none (the
    head and the tail of the row): the first index whose running sum, slice by
    slice, reaches the target."""
    ms = gpu
    say(f"sample flat tail V={V}")
    dh = ms.DeviceBuffer.from_array(np.zeros(1, np.int32))
    v = np.full(V, -6.0, np.float32)
    v[V // 2] = 18.0 + np.log(V)
    dl = ms.DeviceBuffer(V * 4)
    per = (V + 1023) // 1024
    targets = sorted((oracle.sample_target(s), s) for s in range(400000))
    for t, seed in targets[:6] + targets[200000:200002] + targets[-6:]:
        dl.upload(v)
        gid = ms.sample(dl, V, 1.0, dh, 0, 1.0, seed)
        p = dl.download(np.float32, V)
        want, base = V - 1, np.float32(0)
        for c in range(0, V, per):
            run = base + np.zeros(1, np.float32)
            cum = np.cumsum(np.concatenate([run, p[c:c + per]]), dtype=np.float32)[1:]
            hit = np.flatnonzero(cum >= np.float32(t))
            if hit.size:
                want = c + int(hit[0])
                break
            base = np.float32(base + np.cumsum(p[c:c + per], dtype=np.float32)[-1])
        assert gid == want, (t, gid, want)
    dl.free()
    dh.free()
