"""The prefill GEMM (more than 16 rows) through ms_q4_matmul at the edges of its
tiles: 32 or 64 rows by 8 to 16 panels, with and without a split of K.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"\n[case] {msg}", flush=True)


def _matmul(ms, a, w, K, N, scale, c0=None):
    M = a.shape[0]
    dA = ms.DeviceBuffer.from_array(a)
    dC = ms.DeviceBuffer.from_array(c0 if c0 is not None else np.zeros((M, N), np.float32))
    ms.check(ms.lib().ms_q4_matmul(dC.ptr, dA.ptr, w.ptr, M, K, N, C.c_float(scale),
                                   1 if c0 is not None else 0))
    out = dC.download(np.float32, (M, N))
    dA.free()
    dC.free()
    return out


# (M, K, N): rows and columns at, below and above the tiles' edges; one round of
# blocks, several, and remainders; K from one step on, K parts of unequal length
CASES = [(17, 128, 16), (31, 256, 144), (33, 384, 272), (64, 128, 2560), (65, 2560, 160),
         (63, 10240, 272), (33, 1664, 5136), (129, 4224, 1040), (257, 256, 20480),
         (511, 256, 6160), (513, 128, 3088), (1000, 256, 5120), (1025, 128, 8208),
         (2047, 128, 2576), (2049, 256, 3072)]


@pytest.mark.parametrize("M,K,N", CASES)
def test_gemm_tile_edges(gpu, M, K, N):
    """Against 64 bits: 22-bit rows are within 2^-23 of their maximum per value, so
    an output is off by at most 2^-23 max|a_row| sum_k |w_k| (plus its own fp32
    rounding).  Rows do not depend on the launch: the last 17 alone (another tile,
    another split) give the same bits.  Accumulating adds to what is there."""
    ms = gpu
    say(f"gemm edges M={M} K={K} N={N}")
    rng = np.random.default_rng(M * 31 + K + N)
    raw = rng.integers(0, 256, (K, N // 2)).astype(np.uint8)
    scale = np.float32(0.03)
    dr = ms.DeviceBuffer.from_array(raw)
    w = ms.DeviceBuffer(K * N // 2)
    ms.check(ms.lib().ms_q4_pack(w.ptr, dr.ptr, K, N))
    a = rng.standard_normal((M, K)).astype(np.float32)
    got = _matmul(ms, a, w, K, N, scale)
    deq = np.empty((K, N), np.float64)
    deq[:, 0::2] = (raw & 15).astype(np.float64) - 8
    deq[:, 1::2] = (raw >> 4).astype(np.float64) - 8
    deq *= float(scale)
    ref = a.astype(np.float64) @ deq
    bound = (2.0 ** -23) * np.abs(a).max(1)[:, None] * np.abs(deq).sum(0)[None] + \
        2.0 ** -23 * np.abs(ref)
    assert np.all(np.abs(got - ref) <= bound)
    assert np.array_equal(_matmul(ms, a[-17:].copy(), w, K, N, scale), got[-17:])
    acc = _matmul(ms, a, w, K, N, scale, got)
    assert np.array_equal(acc, got + got)
    dr.free()
    w.free()
