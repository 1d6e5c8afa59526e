"""Q4 products of 5 to 16 rows (limbs in MFMA fragment order, k_gemv_rows) at the
edges of its row groups, panels per block, waves and batches of K.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"\n[case] {msg}", flush=True)


# (M, K, N): 4, 8 and 16 waves; one super-tile in all, fewer than waves, one
# batch, several with a remainder; one and two panels per block, odd panels
CASES = [(5, 128, 16), (6, 256, 32), (8, 640, 48), (9, 2560, 3072), (13, 2560, 10240),
         (7, 2688, 16400), (16, 10240, 2560), (12, 13824, 160), (16, 16384, 16),
         (11, 5120, 16448), (15, 3712, 20480), (8, 384, 4096)]


def _weights(ms, rng, K, N):
    raw = rng.integers(0, 256, (K, N // 2)).astype(np.uint8)
    dr = ms.DeviceBuffer.from_array(raw)
    w = ms.DeviceBuffer(K * N // 2)
    ms.check(ms.lib().ms_q4_pack(w.ptr, dr.ptr, K, N))
    ms.synchronize()
    dr.free()
    deq = np.empty((K, N), np.float64)
    deq[:, 0::2] = (raw & 15).astype(np.float64) - 8
    deq[:, 1::2] = (raw >> 4).astype(np.float64) - 8
    return w, deq


def _bound(a, deq, ref):
    """31-bit rows: within 2^-30 of their maximum per value; one fp32 rounding."""
    return 2.0 ** -30 * np.abs(a).max(1)[:, None] * np.abs(deq).sum(0)[None] + \
        2.0 ** -23 * np.abs(ref)


@pytest.mark.parametrize("M,K,N", CASES)
def test_rows_edges(gpu, M, K, N):
    """Against 64 bits; the first five rows alone give the same bits; accumulating
    adds to what is there."""
    ms = gpu
    say(f"gemv rows M={M} K={K} N={N}")
    rng = np.random.default_rng(M * 31 + K + N)
    w, deq = _weights(ms, rng, K, N)
    scale = np.float32(0.03)
    a = (rng.standard_normal((M, K)) * np.exp(rng.uniform(-4, 4, (M, 1)))).astype(np.float32)
    a[M // 2] = 0.0

    def run(rows, c0, acc):
        dA = ms.DeviceBuffer.from_array(rows)
        dC = ms.DeviceBuffer.from_array(c0)
        ms.check(ms.lib().ms_q4_matmul(dC.ptr, dA.ptr, w.ptr, len(rows), K, N, C.c_float(scale),
                                       acc))
        out = dC.download(np.float32, c0.shape)
        dA.free()
        dC.free()
        return out

    got = run(a, np.zeros((M, N), np.float32), 0)
    deq *= float(scale)
    ref = a.astype(np.float64) @ deq
    assert np.all(np.abs(got - ref) <= _bound(a, deq, ref))
    assert np.array_equal(run(a[:5].copy(), np.zeros((5, N), np.float32), 0), got[:5])
    assert np.array_equal(run(a, got, 1), got + got)
    w.free()


@pytest.mark.parametrize("M", [5, 8, 9, 16])
def test_rows_head(gpu, M):
    """The head's logits and first maxima of 5 to 16 rows."""
    ms = gpu
    K, N = 1024, 64 * 33
    say(f"head rows M={M}")
    rng = np.random.default_rng(M)
    w, deq = _weights(ms, rng, K, N)
    scale = np.float32(0.02)
    a = rng.standard_normal((M, K)).astype(np.float32)
    dA = ms.DeviceBuffer.from_array(a)
    dL, dI = ms.DeviceBuffer(M * N * 4), ms.DeviceBuffer(M * 4)
    ms.check(ms.lib().ms_lm_head_argmax(dA.ptr, M, K, w.ptr, N, C.c_float(scale), dL.ptr, dI.ptr))
    got = dL.download(np.float32, (M, N))
    deq *= float(scale)
    ref = a.astype(np.float64) @ deq
    assert np.all(np.abs(got - ref) <= _bound(a, deq, ref))
    assert np.array_equal(dI.download(np.int32, M), got.argmax(1))
    for b in (dA, dL, dI, w):
        b.free()
