"""Prefill attention (flash.hip) against a float64 statement of causal GQA:
numbers of query heads per kv head that do not divide the 64-query tiles, every
head size, rows and positions at the edges of the 32-key tiles, key splits, a
window shorter than the rows, and the cache contents afterwards.

Bound: q, k, v and p enter exactly (three bf16 parts), each product lacks less than
2^-24 of itself, sums are fp32.  A score's error is then below about 3 * 2^-24 * sum |q
k| scale, at |q|, |k| ~ 2 and hd <= 512 below 1e-5 absolute, and moves a probability by
as much relatively; the outputs' relative RMSE is held to 2e-6 (an fp32 evaluation shows
1e-7 .. 5e-7)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# name, heads, kv heads, head dim, circular, cache_len, clamp, T, base
CASES = [
    ("g5-first-tile", 10, 2, 128, 0, 256, 0, 17, 0),
    ("g5-tile-edge", 10, 2, 128, 0, 256, 0, 32, 0),
    ("g5-one-past", 10, 2, 128, 0, 256, 0, 33, 31),
    ("g5-long", 10, 2, 128, 0, 1100, 0, 1000, 64),
    ("g1", 2, 2, 128, 0, 256, 0, 65, 3),
    ("g3-circular", 6, 2, 256, 1, 96, 0, 130, 50),
    ("g4-window", 8, 2, 256, 1, 512, 0, 700, 0),
    ("g20", 20, 1, 128, 1, 64, 0, 45, 200),
    ("hd64", 8, 2, 64, 0, 512, 0, 300, 7),
    ("hd512-split", 8, 2, 512, 0, 1024, 1, 600, 0),
    ("hd512-clamp", 8, 2, 512, 0, 128, 1, 40, 100),
    ("hd512-past-cache", 8, 2, 512, 0, 128, 1, 20, 300),
]


def reference(q, k, v, G, lo, hi, key0):
    """q [T][nh][hd], k and v [keys][nkv][hd] at positions key0 .."""
    T, nh, hd = q.shape
    out = np.empty_like(q)
    for h in range(nh):
        s = q[:, h] @ k[:, h // G].T / np.sqrt(hd)
        p = key0 + np.arange(k.shape[0])
        s[(p[None] < lo[:, None]) | (p[None] > hi[:, None])] = -np.inf
        e = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = (e / e.sum(1, keepdims=True)) @ v[:, h // G]
    return out


@pytest.mark.parametrize("scale", [1.0, 1e-3, 300.0])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_prefill_attention(gpu, case, scale):
    ms = gpu
    name, nh, nkv, hd, circ, clen, clamp, T, base = case
    print(f"[flash] {name} T={T} base={base} scale={scale}", flush=True)
    rng = np.random.default_rng(T * 7 + base)
    qd, kvd, G = nh * hd, nkv * hd, nh // nkv
    kc = (rng.standard_normal((clen, kvd)) * 2).astype(np.float32)
    # v of different size by position, and k and q whose product keeps its size
    vc = (rng.standard_normal((clen, kvd)) * scale).astype(np.float32)
    q = (rng.standard_normal((T, qd)) * 2 / scale).astype(np.float32)
    kc *= np.float32(scale)
    kn = (rng.standard_normal((T, kvd)) * 2 * scale).astype(np.float32)
    vn = (rng.standard_normal((T, kvd)) * scale * np.exp2(rng.integers(-3, 4, (T, 1)))).astype(
        np.float32)
    desc = ms.LayerDesc(q_dim=qd, kv_dim=kvd, head_dim=hd, n_heads=nh, n_kv_heads=nkv,
                        rot_dim=hd, theta=1e4, cache_kind=circ, cache_len=clen,
                        clamp_reads=clamp)
    pos = base + np.arange(T)
    lo = np.maximum(0, pos - clen + 1) if circ else np.zeros(T, int)
    hi = np.minimum(pos, clen - 1) if clamp else pos
    k0 = int(lo[0])
    old = np.arange(k0, min(base, base if circ else clen))
    slot = old % clen if circ else old
    k = np.concatenate([kc[slot], kn]).astype(np.float64)
    v = np.concatenate([vc[slot], vn]).astype(np.float64)
    if not circ and base > clen:  # nothing of the rows is attended
        k, v = k[:clen], v[:clen]
    ref = reference(q.astype(np.float64).reshape(T, nh, hd), k.reshape(-1, nkv, hd),
                    v.reshape(-1, nkv, hd), G, lo, hi, k0).reshape(T, qd)
    dq, dk, dv = (ms.DeviceBuffer.from_array(a) for a in (q, kn, vn))
    dkc, dvc = ms.DeviceBuffer.from_array(kc), ms.DeviceBuffer.from_array(vc)
    dout = ms.DeviceBuffer(T * qd * 4)
    ms.check(ms.lib().ms_attention(C.byref(desc), dq.ptr, dk.ptr, dv.ptr, dkc.ptr, dvc.ptr, T,
                                   base, dout.ptr))
    got = dout.download(np.float32, (T, qd)).astype(np.float64)
    err = np.sqrt(np.mean((got - ref) ** 2) / np.mean(ref ** 2))
    print(f"[flash]   rel rmse {err:.2e}", flush=True)
    assert err < 2e-6
    wk, wv = kc.copy(), vc.copy()
    for r in range(T):
        s = (base + r) % clen if circ else base + r
        if s < clen:
            wk[s], wv[s] = kn[r], vn[r]
    assert np.array_equal(dkc.download(np.float32, kc.shape), wk)
    assert np.array_equal(dvc.download(np.float32, vc.shape), wv)


def test_prefill_attention_nan_row_stays_in_its_tile(gpu):
    """A NaN in the last row's q reaches no other row; an all-zero k or v tile
    gives the mean of v, or zero."""
    ms = gpu
    T, nh, nkv, hd = 70, 5, 1, 128
    rng = np.random.default_rng(3)
    q = rng.standard_normal((T, nh * hd)).astype(np.float32)
    q[-1, 5] = np.nan
    kn = np.zeros((T, hd), np.float32)
    vn = rng.standard_normal((T, hd)).astype(np.float32)
    vn[:64] = 0
    desc = ms.LayerDesc(q_dim=nh * hd, kv_dim=hd, head_dim=hd, n_heads=nh, n_kv_heads=nkv,
                        rot_dim=hd, theta=1e4, cache_kind=0, cache_len=128, clamp_reads=0)
    dq, dk, dv = (ms.DeviceBuffer.from_array(a) for a in (q, kn, vn))
    dkc, dvc = (ms.DeviceBuffer.from_array(np.zeros((128, hd), np.float32)) for _ in "kv")
    dout = ms.DeviceBuffer(T * nh * hd * 4)
    ms.check(ms.lib().ms_attention(C.byref(desc), dq.ptr, dk.ptr, dv.ptr, dkc.ptr, dvc.ptr, T, 0,
                                   dout.ptr))
    got = dout.download(np.float32, (T, nh, hd))
    mean = np.cumsum(vn.astype(np.float64), 0) / np.arange(1, T + 1)[:, None]
    assert np.array_equal(got[:64], np.zeros((64, nh, hd), np.float32))
    assert np.abs(got[:-1] - mean[:-1, None]).max() < 1e-6
    assert np.abs(got[-1, 1:] - mean[-1]).max() < 1e-6
    assert np.isnan(got[-1, 0]).all()


def attend(ms, nh, nkv, hd, circ, clen, q, kn, vn, base=0):
    """ms_attention on fresh rows after zero caches (base 0)."""
    T = len(q)
    desc = ms.LayerDesc(q_dim=nh * hd, kv_dim=nkv * hd, head_dim=hd, n_heads=nh, n_kv_heads=nkv,
                        rot_dim=hd, theta=1e4, cache_kind=circ, cache_len=clen, clamp_reads=0)
    bufs = [ms.DeviceBuffer.from_array(np.ascontiguousarray(a.reshape(T, -1), np.float32))
            for a in (q, kn, vn)]
    caches = [ms.DeviceBuffer.from_array(np.zeros((clen, nkv * hd), np.float32)) for _ in "kv"]
    out = ms.DeviceBuffer(T * nh * hd * 4)
    ms.check(ms.lib().ms_attention(C.byref(desc), *(b.ptr for b in bufs + caches), T, base,
                                   out.ptr))
    got = out.download(np.float32, (T, nh, hd))
    for b in bufs + caches + [out]:
        b.free()
    return got


SPREADS = [("k-row", 128), ("k-row", 512), ("v-row", 256), ("v-row", 512), ("v-dims", 64),
           ("v-dims", 256), ("v-dims", 512), ("k-dims", 128), ("k-dims", 512)]


@pytest.mark.parametrize("kind,hd", SPREADS)
def test_prefill_attention_magnitudes(gpu, kind, hd):
    """Values 2^24 apart in one tile: a key, or a value, of no weight beside ordinary
    ones, and dims of very different size.  Every row, head and dim is held to the
    error of an fp32 evaluation by itself: the operands are exact and a sum of n
    products in fp32 is off by about sqrt(n) 2^-25 of its terms' 2-norm, below 1e-6 here
    for the scores (|s| ~ 1) and the outputs."""
    ms = gpu
    T, nh, nkv = 150, 4, 2
    print(f"[flash] magnitudes {kind} hd={hd}", flush=True)
    rng = np.random.default_rng(hd)
    q = rng.standard_normal((T, nh, hd))
    k = rng.standard_normal((T, nkv, hd))
    v = rng.standard_normal((T, nkv, hd)) + 0.5
    big = 2.0 ** 24
    if kind in ("k-row", "v-row"):
        # key 40 scores far below every other and has no weight
        q[:, :, 0] = np.abs(q[:, :, 0]) + 1
        k[40] = 0
        k[40, :, 0] = -big if kind == "k-row" else -2000.0 * np.sqrt(hd)
        if kind == "v-row":
            v[40] *= big
        rows = np.r_[0:40, 41:T]  # (row 40's first keys are ordinary as well)
    else:
        f = np.exp2(24.0 * np.arange(hd) / hd - 12).astype(np.float32)
        if kind == "v-dims":
            v *= f
        else:
            k, q = k * f, q / f
        rows = np.arange(T)
    q, k, v = (a.astype(np.float32) for a in (q, k, v))
    got = attend(ms, nh, nkv, hd, 0, 256, q, k, v).astype(np.float64)
    pos = np.arange(T)
    ref = reference(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), nh // nkv,
                    np.zeros(T, int), pos, 0)
    e, r = (got - ref)[rows], ref[rows]
    row_err = np.sqrt((e ** 2).mean(2) / (r ** 2).mean(2))
    dim_err = np.sqrt((e ** 2).mean(0) / (r ** 2).mean(0))
    print(f"[flash]   worst row {row_err.max():.2e}, worst dim {dim_err.max():.2e}", flush=True)
    if kind != "v-dims":
        assert row_err.max() < 2e-6
    assert dim_err.max() < 2e-6


@pytest.mark.parametrize("hd", [64, 128, 256, 512])
def test_prefill_attention_rows_do_not_depend_on_later_ones(gpu, hd):
    """Later rows change no bit of an earlier row's output, whatever their size."""
    ms = gpu
    rng = np.random.default_rng(hd)
    T, nh, nkv = 70, 4, 2
    q, k, v = (rng.standard_normal((T, n, hd)).astype(np.float32) for n in (nh, nkv, nkv))
    a = attend(ms, nh, nkv, hd, 0, 128, q, k, v)
    for r in (5, 37, 69):
        k2, v2 = k.copy(), v.copy()
        k2[r:] *= np.float32(3e4)
        v2[r:] *= np.float32(3e-5)
        b = attend(ms, nh, nkv, hd, 0, 128, q, k2, v2)
        assert np.array_equal(a[:r], b[:r])


@pytest.mark.parametrize("hd,T", [(64, 70), (128, 150), (256, 300), (512, 600)])
@pytest.mark.parametrize("kind", ["v-nan", "v-inf", "k-inf", "k-weightless"])
def test_prefill_attention_not_finite(gpu, kind, hd, T):
    """A value that is not finite reaches the rows that attend to its key with a weight,
    in its dim, and no other: not earlier rows of its tile, and not through the parts of
    the operands.  (The last case has keys in several splits.)"""
    ms = gpu
    print(f"[flash] {kind} hd={hd} T={T}", flush=True)
    nh, nkv, r = 4, 2, T // 2 + 9
    rng = np.random.default_rng(hd)
    q, k, v = (rng.standard_normal((T, n, hd)).astype(np.float32) for n in (nh, nkv, nkv))
    q[:, :, 3] = np.abs(q[:, :, 3]) + np.float32(0.1)
    pos = np.arange(T)
    zero = np.zeros(T, int)
    f64 = [a.astype(np.float64) for a in (q, k, v)]
    if kind == "k-weightless":
        # a score of -inf in kv head 1: the same as without the key
        k[r, 1, 3] = -np.inf
        ref = reference(*f64, nh // nkv, zero, pos, 0)
        rest = np.delete(pos, r)
        with_r = reference(f64[0][r:], f64[1][rest], f64[2][rest], nh // nkv, zero[r:],
                           pos[r:] - 1, 0)
        ref[r:, 2:] = with_r[:, 2:]
        hit = np.zeros((T, nh, hd), bool)
        value = None
    else:
        ref = reference(*f64, nh // nkv, zero, pos, 0)
        hit = np.zeros((T, nh, hd), bool)
        if kind == "k-inf":
            k[r, 1, 3] = np.inf  # the softmax of an infinite score: NaN
            hit[r:, 2:] = True
            value = np.isnan
        else:
            v[r, 1, 5] = np.nan if kind == "v-nan" else np.inf
            hit[r:, 2:, 5] = True
            value = np.isnan if kind == "v-nan" else np.isposinf
    got = attend(ms, nh, nkv, hd, 0, 1024, q, k, v)
    if value is not None:
        assert value(got[hit]).all()
    e, w = got[~hit] - ref[~hit], ref[~hit]
    assert np.isfinite(e).all()
    err = np.sqrt(np.mean(e ** 2) / np.mean(w ** 2))
    print(f"[flash]   rel rmse {err:.2e}", flush=True)
    assert err < 2e-6


def test_prefill_attention_not_finite_outside_the_window(gpu):
    """Cached keys that the window has left, in the first tile of the rows, are not
    finite: no row sees them."""
    ms = gpu
    nh, nkv, hd, clen, T, base = 4, 2, 128, 96, 40, 150
    rng = np.random.default_rng(5)
    q, kn, vn = (rng.standard_normal((T, n * hd)).astype(np.float32) for n in (nh, nkv, nkv))
    kc, vc = (rng.standard_normal((clen, nkv * hd)).astype(np.float32) for _ in "kv")
    pos = base + np.arange(T)
    lo = pos - clen + 1
    old = np.arange(lo[0], base)
    # (keys 32 .. 54 share a tile with key 55, the first that a row attends to; their
    # slots now hold keys 128 .. 149 and one that is to come)
    slot = (lo[0] - 1) % clen
    kc[slot], vc[slot] = np.nan, np.inf
    k = np.concatenate([kc[old % clen], kn]).astype(np.float64).reshape(-1, nkv, hd)
    v = np.concatenate([vc[old % clen], vn]).astype(np.float64).reshape(-1, nkv, hd)
    ref = reference(q.astype(np.float64).reshape(T, nh, hd), k, v, nh // nkv, lo, pos, lo[0])
    desc = ms.LayerDesc(q_dim=nh * hd, kv_dim=nkv * hd, head_dim=hd, n_heads=nh, n_kv_heads=nkv,
                        rot_dim=hd, theta=1e4, cache_kind=1, cache_len=clen, clamp_reads=0)
    bufs = [ms.DeviceBuffer.from_array(a) for a in (q, kn, vn, kc, vc)]
    out = ms.DeviceBuffer(T * nh * hd * 4)
    ms.check(ms.lib().ms_attention(C.byref(desc), *(b.ptr for b in bufs), T, base, out.ptr))
    got = out.download(np.float32, (T, nh, hd))
    assert np.isfinite(got).all()
    assert np.sqrt(np.mean((got - ref) ** 2) / np.mean(ref ** 2)) < 2e-6
