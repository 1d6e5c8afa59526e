// Token sampling on the device: temperature_sampling (lm_head.mojo:198-254)
// with a caller-given seed where the reference reads the clock (:246).
//
// A row is kSampleSlices contiguous slices; blocks of 256 threads own whole
// slices, about kSampleTile logits each, so that a row of a large vocabulary
// spreads over the chip (262144 logits: 128 blocks).  Every intermediate is
// written back in place as in the reference, four launches over the row:
//   k_sample_max   penalty and maximum.  Each id of the row's history that is
//                  below n, once per occurrence: a positive logit divided by
//                  the penalty, any other multiplied (:211-220).  A block
//                  counts the occurrences of its own ids in LDS and applies
//                  the operation that many times, which is the reference's
//                  sequence of operations on that logit.
//   k_sample_pass  exp((v - max) / T) and the slices' sums (:230-238); launched
//                  again, the division by the sum (:239-243) and the slices'
//                  new sums
//   k_sample_draw  one LCG step of the seed (:246-248; in the model the seed
//                  of draw k of sequence b is draw_seed(seed, b, k)); the first
//                  index whose running sum reaches the target, else n - 1
//                  (:250-254).
// Greedy (temperature <= 0.01, :222-228) takes the first index of the maximum
// from k_sample_max's block maxima.
//
// A slice's sum adds its values in order and the slices' sums are added in
// slice order, so the result does not depend on the blocks.  The sums round
// differently from the reference's one running sum, so a draw whose target
// lies within rounding of a slice boundary of the cumulative distribution may
// pick the neighbouring index.
//
// Bound by latency: the launches and, in each, one chain of additions (a
// slice's 256 values, or the 1024 slices' sums).  262144 logits, 600 ids of
// history: 37 to 39 us for the four; one block per row took 878 us.
#include "common.h"
#include "sample.h"

#include <cmath>

namespace ms {
namespace {

constexpr int kSampleTile = 2048;  // logits per pass of a block
constexpr int kSampleNT = 256;
// LDS position of value i of a tile whose slices are `per` long: one word of
// padding per slice, so that the threads adding different slices read
// different banks
__device__ inline int pad_pos(int i, int per) { return i + i / per; }

template <class T>
__device__ inline T sld(const T *p) {
  return *(const __attribute__((address_space(1))) T *)p;
}

// lm_head.mojo:247-248 in wrapping 64-bit arithmetic
__device__ inline float lcg_target(uint64_t seed) {
  const uint64_t lcg = (seed * 6364136223846793005ull + 1442695040888963407ull) & 0x7FFFFFFFull;
  return (float)lcg / (float)0x7FFFFFFF;
}

// Logits per slice and slices per block of a row of n logits.
__host__ __device__ inline int slice_len(int n) { return (n + kSampleSlices - 1) / kSampleSlices; }
__host__ __device__ inline int block_slices(int n) {
  const int s = kSampleTile / slice_len(n);
  return s < 1 ? 1 : s < kSampleNT ? s : kSampleNT;
}
__host__ __device__ inline int row_blocks(int n) {
  return (kSampleSlices + block_slices(n) - 1) / block_slices(n);
}
// Workspace of a row: block maxima and their indices, slice sums of the
// exponentials and of the probabilities.
__device__ inline float *row_work(const SampleArgs &a, int row) {
  return a.work + (size_t)row * 4 * kSampleSlices;
}

// The larger value, the lower index among equals; a NaN never wins.
__device__ inline void max_first(float &m, int &mi, float v, int i) {
  if (v > m || (v == m && i < mi)) {
    m = v;
    mi = i;
  }
}
template <int NT>
__device__ inline void block_max_first(float &m, int &mi, float *rv, int *ri) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float ov = __shfl_xor(m, o, 64);
    const int oi = __shfl_xor(mi, o, 64);
    max_first(m, mi, ov, oi);
  }
  if ((threadIdx.x & 63) == 0) {
    rv[threadIdx.x >> 6] = m;
    ri[threadIdx.x >> 6] = mi;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) max_first(m, mi, rv[w], ri[w]);
}

__global__ __launch_bounds__(kSampleNT) void k_sample_max(SampleArgs a) {
  __shared__ int cnt[kSampleTile];
  __shared__ float rv[kSampleNT / 64];
  __shared__ int ri[kSampleNT / 64];
  const int tid = threadIdx.x, row = blockIdx.y, n = a.n;
  const int per = slice_len(n), spb = block_slices(n);
  float *v = a.logits + (size_t)row * a.ld;
  const bool pen = a.penalty > 1.0f && a.hist;
  const int32_t *h = a.hist + (size_t)row * a.hist_ld;
  const int nh = !pen ? 0 : min(a.hist_n ? sld(a.hist_n + row) : a.hist_len, kSampleMaxHistory);
  const long b0 = (long)blockIdx.x * spb * per;
  const int e0 = (int)min((long)n, b0), e1 = (int)min((long)n, b0 + (long)spb * per);
  float m = -INFINITY;
  int mi = n;
  for (int t0 = e0; t0 < e1; t0 += kSampleTile) {
    const int nt = min(kSampleTile, e1 - t0);
    if (nh > 0) {
      __syncthreads();
      for (int i = tid; i < nt; i += kSampleNT) cnt[i] = 0;
      __syncthreads();
      for (int i = tid; i < nh; i += kSampleNT) {
        const unsigned p = (unsigned)sld(h + i) - (unsigned)t0;
        if (p < (unsigned)nt) atomicAdd(&cnt[p], 1);
      }
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < kSampleTile / kSampleNT; ++j) {
      const int i = j * kSampleNT + tid;
      if (i >= nt) continue;
      float x = sld(v + t0 + i);
      if (nh > 0 && cnt[i] > 0) {
        for (int k = cnt[i]; k > 0; --k) x = x > 0.0f ? x / a.penalty : x * a.penalty;
        v[t0 + i] = x;
      }
      max_first(m, mi, x, t0 + i);
    }
  }
  block_max_first<kSampleNT>(m, mi, rv, ri);
  if (tid == 0) {
    if (blockIdx.x == 0) {
      const float x = v[0];
      if (x != x) m = x;
    }
    float *w = row_work(a, row);
    w[blockIdx.x] = m;
    reinterpret_cast<int *>(w + kSampleSlices)[blockIdx.x] = mi;
  }
}

// Maximum of the row and its first index (a NaN in front is the maximum, as
// for the reference's scan; no logit above -inf: index 0).
template <int NT>
__device__ inline void row_max(const SampleArgs &a, int row, float *rv, int *ri, float *vmax,
                               int *imax) {
  const float *w = row_work(a, row);
  const int *wi = reinterpret_cast<const int *>(w + kSampleSlices);
  float m = -INFINITY;
  int mi = a.n;
  const int nb = row_blocks(a.n);
  for (int i = threadIdx.x; i < nb; i += NT) max_first(m, mi, sld(w + i), sld(wi + i));
  block_max_first<NT>(m, mi, rv, ri);
  const float w0 = sld(w);
  *vmax = w0 == w0 ? m : w0;
  *imax = w0 == w0 && mi < a.n ? mi : 0;
}

// NORM false: v = exp((v - max) / T); true: v = v / (sum of the exponentials).
// Either way the sums of the block's slices of the new values.
template <bool NORM>
__global__ __launch_bounds__(kSampleNT) void k_sample_pass(SampleArgs a) {
  __shared__ float t[kSampleTile + kSampleSlices];
  __shared__ float rv[kSampleNT / 64], total;
  __shared__ int ri[kSampleNT / 64];
  const int tid = threadIdx.x, row = blockIdx.y, n = a.n;
  const int per = slice_len(n), spb = block_slices(n);
  float *v = a.logits + (size_t)row * a.ld;
  float *w = row_work(a, row);
  const long b0 = (long)blockIdx.x * spb * per;
  const int e0 = (int)min((long)n, b0), e1 = (int)min((long)n, b0 + (long)spb * per);
  float x[kSampleTile / kSampleNT];
  auto load = [&](int t0) {
#pragma unroll
    for (int j = 0; j < kSampleTile / kSampleNT; ++j) {
      const int i = t0 + j * kSampleNT + tid;
      x[j] = i < e1 ? sld(v + i) : 0.f;
    }
  };
  load(e0);  // beside the reduction below
  float f = 0.f;
  if constexpr (NORM) {
    for (int i = tid; i < kSampleSlices; i += kSampleNT) t[i] = sld(w + 2 * kSampleSlices + i);
    __syncthreads();
    if (tid == 0) {
      float z = 0.0f;
#pragma unroll 32
      for (int i = 0; i < kSampleSlices; ++i) z += t[i];
      total = z;
    }
    __syncthreads();
    f = 1.0f / total;
  } else {
    int imax;
    row_max<kSampleNT>(a, row, rv, ri, &f, &imax);
  }
  const float inv_t = 1.0f / a.temperature;
  float s = 0.f;
  for (int t0 = e0; t0 < e1; t0 += kSampleTile) {
    // (a block of several slices has one tile)
    const int nt = min(kSampleTile, e1 - t0);
    if (t0 > e0) load(t0);
#pragma unroll
    for (int j = 0; j < kSampleTile / kSampleNT; ++j) {
      const int i = j * kSampleNT + tid;
      if (i >= nt) continue;
      const float y = NORM ? x[j] * f : expf((x[j] - f) * inv_t);
      v[t0 + i] = y;
      t[pad_pos(i, per)] = y;
    }
    __syncthreads();
    if (tid < spb) {
      const int len = min(per, nt - tid * per);
      const float *q = t + tid * (per + 1);
#pragma unroll 16
      for (int i = 0; i < len; ++i) s += q[i];
    }
    __syncthreads();
  }
  const int sl = blockIdx.x * spb + tid;
  if (tid < spb && sl < kSampleSlices) w[(NORM ? 3 : 2) * kSampleSlices + sl] = s;
}

__global__ __launch_bounds__(kSampleSlices) void k_sample_draw(SampleArgs a) {
  constexpr int NT = kSampleSlices;
  __shared__ float part[NT], sum[NT], rv[NT / 64];
  __shared__ int ri[NT / 64];
  const int tid = threadIdx.x, row = blockIdx.x, n = a.n;
  const float *v = a.logits + (size_t)row * a.ld;
  int result;
  if (a.temperature <= 0.01f) {
    float vmax;
    row_max<NT>(a, row, rv, ri, &vmax, &result);
  } else {
    const float lp = sld(row_work(a, row) + 3 * kSampleSlices + tid);
    part[tid] = lp;
    __syncthreads();
    if (tid == 0) {
      // (out of place, so that the reads run ahead of the writes)
      float z = 0.0f;
#pragma unroll 32
      for (int i = 0; i < NT; ++i) {
        sum[i] = z;
        z += part[i];
      }
    }
    __syncthreads();
    const uint64_t seed =
        a.step ? draw_seed(a.seed, (uint64_t)(a.seq0 + row), (uint64_t)sld(a.step)) : a.seed;
    const float target = lcg_target(seed);
    const int per = slice_len(n);
    const int c0 = (int)min((long)n, (long)tid * per), c1 = (int)min((long)n, (long)c0 + per);
    float cdf = sum[tid];
    int found = n;
    // Only a slice whose sum comes within rounding of the target is walked:
    // each of its additions, to a running sum of at most about one, is off by
    // 2^-24 at most, and so is each of the slice sum's.
    if (c0 < c1 && cdf >= target) {
      found = c0;
    } else if (cdf + lp >= target - (float)(per + 8) * 0x1p-22f) {
      // (32 loads in flight: a walk of 256 values is a chain of eight)
      for (int j0 = c0; j0 < c1 && found == n; j0 += 32) {
        float x[32];
#pragma unroll
        for (int j = 0; j < 32; ++j) x[j] = sld(v + min(j0 + j, c1 - 1));
#pragma unroll
        for (int j = 0; j < 32; ++j) {
          cdf += x[j];
          if (j0 + j < c1 && found == n && cdf >= target) found = j0 + j;
        }
      }
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) found = min(found, __shfl_xor(found, o, 64));
    if ((tid & 63) == 0) ri[tid >> 6] = found;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) found = min(found, ri[i]);
    result = found < n ? found : n - 1;
  }
  if (tid == 0) {
    if (a.ids_out) a.ids_out[row] = result;
    if (a.tok_state) a.tok_state[row] = result;
    if (a.hist_append) {
      // the sampled id joins the row's history for the next draw
      const int nh = sld(a.hist_n + row);
      if (nh < a.hist_cap) a.hist[(size_t)row * a.hist_ld + nh] = result;
      a.hist_n[row] = min(nh + 1, a.hist_cap);
    }
  }
}

}  // namespace

int launch_sample(const SampleArgs &a, int rows, hipStream_t st) {
  MS_CHECK_ARG(a.logits && a.n >= 1 && a.ld >= a.n && rows >= 1, "sample: bad logits");
  MS_CHECK_ARG(a.temperature == a.temperature && a.penalty == a.penalty,
               "sample: temperature and penalty must be numbers");
  MS_CHECK_ARG(!(a.penalty > 1.0f) || a.hist,
               "sample: a penalty needs the token history");
  MS_CHECK_ARG(a.work, "sample: workspace missing");
  const dim3 grid(row_blocks(a.n), rows), blk(kSampleNT);
  hipLaunchKernelGGL(k_sample_max, grid, blk, 0, st, a);
  if (a.temperature > 0.01f) {
    hipLaunchKernelGGL(k_sample_pass<false>, grid, blk, 0, st, a);
    hipLaunchKernelGGL(k_sample_pass<true>, grid, blk, 0, st, a);
  }
  hipLaunchKernelGGL(k_sample_draw, dim3(rows), dim3(kSampleSlices), 0, st, a);
  MS_HIP_TRY(hipGetLastError());
  return MS_OK;
}

}  // namespace ms

using namespace ms;

extern "C" int ms_sample(float *d_logits, int vocab, float temperature,
                         const int32_t *d_generated, int n_generated, float penalty,
                         uint64_t seed, int32_t *h_id) {
  if (int rc = require_init()) return rc;
  MS_CHECK_ARG(d_logits && vocab >= 1 && h_id, "sample: null argument or empty vocab");
  MS_CHECK_ARG(n_generated >= 0 && n_generated <= kSampleMaxHistory,
               "sample: history longer than 8192 ids");
  MS_CHECK_ARG(n_generated == 0 || d_generated, "sample: history pointer missing");
  hipStream_t st = ctx().stream;
  void *buf = nullptr;
  if (int rc = scratch(kSampleWorkFloats * 4, &buf)) return rc;
  // (a single draw: the seed goes to the LCG step as given); the id comes back
  // through pinned memory, which the kernel's end makes visible
  SampleArgs a{};
  a.work = static_cast<float *>(buf);
  a.logits = d_logits;
  a.n = vocab;
  a.ld = vocab;
  a.temperature = temperature;
  a.penalty = penalty;
  a.hist = const_cast<int32_t *>(d_generated);
  a.hist_ld = n_generated;
  a.hist_len = n_generated;
  a.seed = seed;
  a.ids_out = static_cast<int32_t *>(ctx().host_box);
  if (int rc = launch_sample(a, 1, st)) return rc;
  MS_HIP_TRY(hipStreamSynchronize(st));
  *h_id = *static_cast<volatile int32_t *>(ctx().host_box);
  return MS_OK;
}

extern "C" uint64_t ms_sample_seed(uint64_t seed, int seq, uint64_t draw) {
  return draw_seed(seed, (uint64_t)seq, draw);
}
