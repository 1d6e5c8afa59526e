// Converter quantization on the device: quantize_q4_blockwise
// (scripts/convert.py:296-323) applied to a HuggingFace (out, in) weight, as the
// converter does after its transpose (convert.py:503-518).
//
// The reference transposes to (in, out), splits the flat array into blocks of
// block_size, takes max|w| / 7 per block (1e-8 for a block whose max is not
// above 1e-8) and keeps the largest as the one global scale.  Then
// q = clip(round_half_even(w / scale), -8, 7) + 8, even columns in the low
// nibble.  The largest block scale is max|w| / 7 unless that is below 1e-8 and
// some block is "tiny"; only then does the block structure matter, and only
// then is it examined (k_tiny_blocks).
//
// k_absmax_part  max |w| and a non-finite flag, one pair per block.
// k_q4_pack_t    every block reduces the pairs and forms the scale itself, so
//                that no launch or host round trip stands between the passes; a
//                weight that has to be refused or examined packs nothing and
//                block 0 tells the host.  A thread quantizes 8 rows of 16 bytes
//                in registers (eight loads in flight) and the codes are
//                transposed in LDS as dwords of 8 codes; writes are 128 bytes of
//                an (in, out) row.
//
// Bound by HBM: the weight twice (the second time partly from the last-level
// cache) and half a byte per element written.  bf16 10240 x 2560: 11 + 17.5 us,
// 39 us the call, against 11.7 + 3.4 + 23.6 us of kernels and a copy to the
// host between them, 68 us the call.  The divisions of the former pack kernel
// took most of its time; with the scale's reciprocal a quotient takes five
// operations.
#include "common.h"
#include "devutil.h"

#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace ms {
namespace {

constexpr int kTk = 64;        // in (k) values of a tile
constexpr int kTn = 256;       // out (n) values of a tile of 16-bit weights; fp32: half
constexpr int kRows = 8;       // n values per thread
constexpr int kMaxParts = 1024;

// dtype 0 fp32, 1 bf16, 2 fp16 (SafetensorsReader.load_f32, convert.py:100-110)
__device__ inline float load_w(const void *w, int dtype, size_t i) {
  if (dtype == 0) return static_cast<const float *>(w)[i];
  const uint16_t h = static_cast<const uint16_t *>(w)[i];
  if (dtype == 1) return __uint_as_float((uint32_t)h << 16);
  return __half2float(__ushort_as_half(h));
}

// 16-byte words at element alignment
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
typedef u32x4 u32x4_a1 __attribute__((aligned(1)));

// The 16-byte word v as 4 (fp32) or 8 (bf16, fp16) values.
template <int DT>
__device__ inline void unpack16(const u32x4 v, float *o) {
  const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DT == 0) {
      o[i] = __uint_as_float(u[i]);
    } else if constexpr (DT == 1) {
      o[2 * i] = __uint_as_float(u[i] << 16);
      o[2 * i + 1] = __uint_as_float(u[i] & 0xFFFF0000u);
    } else {
      o[2 * i] = __half2float(__ushort_as_half((uint16_t)(u[i] & 0xFFFFu)));
      o[2 * i + 1] = __half2float(__ushort_as_half((uint16_t)(u[i] >> 16)));
    }
  }
}

// nvec 16-byte words first (the host passes 0 for an unaligned base), then the
// remaining elements one by one.
template <int DT>
__global__ __launch_bounds__(256) void k_absmax_part(const void *w, size_t n, size_t nvec,
                                                     float *part) {
  constexpr int PER = DT == 0 ? 4 : 8;
  __shared__ float sm[256];
  __shared__ int sb[256];
  const int tid = threadIdx.x;
  float m = 0.f;
  int bad = 0;
  const size_t g = (size_t)blockIdx.x * 256 + tid, stride = (size_t)gridDim.x * 256;
  auto take = [&](const u32x4 d) {
    float x[PER];
    unpack16<DT>(d, x);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      bad |= !isfinite(x[i]);
      m = fmaxf(m, fabsf(x[i]));
    }
  };
  size_t v = g;
  for (; v + 3 * stride < nvec; v += 4 * stride) {
    // four loads in flight
    u32x4 d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      d[i] = ldg<u32x4>(static_cast<const uint8_t *>(w) + 16 * (v + i * stride));
#pragma unroll
    for (int i = 0; i < 4; ++i) take(d[i]);
  }
  for (; v < nvec; v += stride) take(ldg<u32x4>(static_cast<const uint8_t *>(w) + 16 * v));
  for (size_t i = nvec * PER + g; i < n; i += stride) {
    const float x = load_w(static_cast<const void *>(w), DT, i);
    bad |= !isfinite(x);
    m = fmaxf(m, fabsf(x));
  }
  sm[tid] = m;
  sb[tid] = bad;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) {
      sm[tid] = fmaxf(sm[tid], sm[tid + s]);
      sb[tid] |= sb[tid + s];
    }
    __syncthreads();
  }
  if (tid == 0) {
    part[2 * blockIdx.x] = sm[0];
    part[2 * blockIdx.x + 1] = (float)sb[0];
  }
}

// flag = 1 when a block of bs consecutive elements of the (in, out) matrix has
// max |w| <= 1e-8 (convert.py:311-314).  Every writer stores the same value.
__global__ __launch_bounds__(256) void k_tiny_blocks(const void *w, int dtype, int n_out, int n_in,
                                                     int bs, size_t nblocks, int *flag) {
  const size_t b = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (b >= nblocks) return;
  const size_t total = (size_t)n_out * n_in;
  const size_t i0 = b * (size_t)bs, i1 = i0 + (size_t)bs < total ? i0 + (size_t)bs : total;
  float m = 0.f;
  for (size_t i = i0; i < i1; ++i) {
    const size_t k = i / (size_t)n_out, o = i % (size_t)n_out;
    m = fmaxf(m, fabsf(load_w(w, dtype, o * (size_t)n_in + k)));
  }
  if (!((double)m > 1e-8)) flag[0] = 1;
}

// clip(round_half_even(x / s), -8, 7) + 8, the quotient rounded to fp32 first as
// the reference's is.  With r = 1 / s correctly rounded, q = x r is within two
// units in the last place of the quotient; q + (x - q s) r is within one, and the
// same step from there gives the correctly rounded quotient (Markstein, IBM J.
// Res. Dev. 34, 1990; the residuals are exact, but for |x| far below s, whose
// code is 8 whatever they are).  Adding 1.5 2^23 rounds half to even.
__device__ inline uint32_t q4_code(float x, float s, float r) {
  float q = x * r;
  q = __builtin_fmaf(__builtin_fmaf(-q, s, x), r, q);
  q = __builtin_fmaf(__builtin_fmaf(-q, s, x), r, q);
  q = __builtin_amdgcn_fmed3f(q, -8.f, 7.f);
  return __float_as_uint(q + (12582912.f + 8.f)) & 15u;
}

// s_given > 0: the scale; else it comes from the npart pairs of k_absmax_part,
// and a non-finite weight or a scale below 1e-8 packs nothing.  Block 0 writes
// (max |w|, flag) to host.  Rows
// of odd lengths start anywhere: the 16-byte words read are element-aligned only,
// and those written at any byte, which the memory unit takes.
template <int DT>
__global__ __launch_bounds__(256) void k_q4_pack_t(const void *w, int n_out, int n_in,
                                                   const float *part, int npart, float s_given,
                                                   float *host, uint8_t *out) {
  constexpr int PER = DT == 0 ? 4 : 8, ESZ = DT == 0 ? 4 : 2;
  constexpr int CPR = kTk / PER;                   // threads along k
  constexpr int TN = 256 / CPR * kRows;            // n values of the tile
  constexpr int LD = TN / 8 + 1;                   // dwords per k row of the tile
  typedef typename std::conditional<DT == 0, u32x4_a4, u32x4_a2>::type Word;
  __shared__ uint32_t t[kTk * LD];
  __shared__ float red[2][4];
  const int tid = threadIdx.x;
  const int k0 = blockIdx.x * kTk, n0 = blockIdx.y * TN;
  const int c = (tid % CPR) * PER, r0 = tid / CPR * kRows;
  u32x4 raw[kRows];
  const bool whole = k0 + c + PER <= n_in;
  auto load = [&]() {
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      raw[i] = u32x4{0, 0, 0, 0};
      if (whole && n0 + r0 + i < n_out)
        raw[i] = *(const __attribute__((address_space(1))) Word *)(
            static_cast<const uint8_t *>(w) + ((size_t)(n0 + r0 + i) * n_in + k0 + c) * ESZ);
    }
  };
  load();
  float s = s_given;
  if (!(s > 0.f)) {
    float m = 0.f, b = 0.f;
    for (int i = tid; i < npart; i += 256) {
      const float2 p = reinterpret_cast<const float2 *>(part)[i];
      m = fmaxf(m, p.x);
      b = fmaxf(b, p.y);
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      m = fmaxf(m, __shfl_xor(m, o, 64));
      b = fmaxf(b, __shfl_xor(b, o, 64));
    }
    if ((tid & 63) == 0) {
      red[0][tid >> 6] = m;
      red[1][tid >> 6] = b;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      m = fmaxf(m, red[0][i]);
      b = fmaxf(b, red[1][i]);
    }
    if (tid == 0 && blockIdx.x == 0 && blockIdx.y == 0) {
      host[0] = m;
      host[1] = b;
    }
    const double gs = (double)m / 7.0;
    if (b != 0.f || !(gs >= 1e-8)) return;
    s = (float)gs;
  }
  const float r = 1.0f / s;
  uint32_t code[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) code[j] = 0;
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    float x[PER];
    unpack16<DT>(raw[i], x);
    if (!whole) {
      // the ragged end of a row, element by element
      for (int j = 0; j < PER; ++j)
        x[j] = n0 + r0 + i < n_out && k0 + c + j < n_in
                   ? load_w(w, DT, (size_t)(n0 + r0 + i) * n_in + k0 + c + j)
                   : 0.f;
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) code[j] |= q4_code(x[j], s, r) << (4 * i);
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) t[(c + j) * LD + r0 / 8] = code[j];
  __syncthreads();
  // 16-byte pieces of the rows
  const size_t half = (size_t)n_out / 2;
#pragma unroll
  for (int e = tid; e < kTk * TN / 32; e += 256) {
    const int kk = e / (TN / 32), p = e % (TN / 32);
    const size_t jb = (size_t)n0 / 2 + 16 * p;
    if (k0 + kk >= n_in || jb >= half) continue;
    const uint32_t *q = t + kk * LD + 4 * p;
    uint8_t *dst = out + (size_t)(k0 + kk) * half + jb;
    if (jb + 16 <= half) {
      *reinterpret_cast<u32x4_a1 *>(dst) = u32x4{q[0], q[1], q[2], q[3]};
    } else {
      for (int j = 0; j < 16 && jb + j < half; ++j) dst[j] = (uint8_t)(q[j / 4] >> (8 * (j % 4)));
    }
  }
}

}  // namespace

}  // namespace ms

using namespace ms;

extern "C" int ms_q4_quantize(uint8_t *d_packed, float *h_scale, const void *d_w, int dtype,
                              int n_out, int n_in, int block_size) {
  if (int rc = require_init()) return rc;
  MS_CHECK_ARG(d_packed && h_scale && d_w, "q4_quantize: null argument");
  MS_CHECK_ARG(dtype >= 0 && dtype <= 2, "q4_quantize: dtype 0 (fp32), 1 (bf16) or 2 (fp16)");
  MS_CHECK_ARG(n_out >= 2 && n_out % 2 == 0 && n_in >= 1,
               "q4_quantize: out dimension must be even (two values per byte, convert.py:304)");
  MS_CHECK_ARG(block_size >= 1, "q4_quantize: block_size must be positive");
  MS_CHECK_ARG((long)n_in <= 65535L * kTk && n_out / 128 < 65535, "q4_quantize: matrix too large");
  hipStream_t st = ctx().stream;
  const size_t n = (size_t)n_out * n_in;
  void *buf = nullptr;
  if (int rc = scratch(kMaxParts * 2 * 4 + 64, &buf)) return rc;
  float *part = static_cast<float *>(buf);
  int *flag = reinterpret_cast<int *>(part + kMaxParts * 2);
  const int esz = dtype == 0 ? 4 : 2, per = 16 / esz;
  const bool aligned = (reinterpret_cast<uintptr_t>(d_w) & 15) == 0;
  const size_t nvec = aligned ? n / per : 0;
  const int nb = (int)std::min<size_t>(kMaxParts, std::max<size_t>(1, cdiv((long)n, 256 * 32)));
  if (dtype == 0)
    hipLaunchKernelGGL(k_absmax_part<0>, dim3(nb), dim3(256), 0, st, d_w, n, nvec, part);
  else if (dtype == 1)
    hipLaunchKernelGGL(k_absmax_part<1>, dim3(nb), dim3(256), 0, st, d_w, n, nvec, part);
  else
    hipLaunchKernelGGL(k_absmax_part<2>, dim3(nb), dim3(256), 0, st, d_w, n, nvec, part);
  float *box = static_cast<float *>(ctx().host_box);
  auto pack = [&](float s) {
    const int tn = dtype == 0 ? kTn / 2 : kTn;
    const dim3 grid(cdiv((long)n_in, kTk), cdiv((long)n_out, tn));
    if (dtype == 0)
      hipLaunchKernelGGL(k_q4_pack_t<0>, grid, dim3(256), 0, st, d_w, n_out, n_in, part, nb, s,
                         box, d_packed);
    else if (dtype == 1)
      hipLaunchKernelGGL(k_q4_pack_t<1>, grid, dim3(256), 0, st, d_w, n_out, n_in, part, nb, s,
                         box, d_packed);
    else
      hipLaunchKernelGGL(k_q4_pack_t<2>, grid, dim3(256), 0, st, d_w, n_out, n_in, part, nb, s,
                         box, d_packed);
  };
  pack(0.f);
  MS_HIP_TRY(hipGetLastError());
  MS_HIP_TRY(hipStreamSynchronize(st));
  const float gmax = reinterpret_cast<volatile float *>(box)[0];
  MS_CHECK_ARG(reinterpret_cast<volatile float *>(box)[1] == 0.f,
               "q4_quantize: the weight holds NaN or infinity");
  // max over the block scales (convert.py:310-316), in double as Python does
  const double g = gmax;
  double gs = g / 7.0;
  if (!(gs >= 1e-8)) {
    // nothing is packed yet
    if (!(g > 1e-8)) {
      gs = 1e-8;  // every block is tiny
    } else {
      const size_t nblocks = (n + block_size - 1) / block_size;
      int tiny = 0;
      MS_HIP_TRY(hipMemcpyAsync(flag, &tiny, 4, hipMemcpyHostToDevice, st));
      hipLaunchKernelGGL(k_tiny_blocks, dim3(cdiv((long)nblocks, 256)), dim3(256), 0, st, d_w,
                         dtype, n_out, n_in, block_size, nblocks, flag);
      MS_HIP_TRY(hipGetLastError());
      MS_HIP_TRY(hipMemcpyAsync(&tiny, flag, 4, hipMemcpyDeviceToHost, st));
      MS_HIP_TRY(hipStreamSynchronize(st));
      if (tiny) gs = 1e-8;
    }
    pack((float)gs);
    MS_HIP_TRY(hipGetLastError());
    MS_HIP_TRY(hipStreamSynchronize(st));
  }
  *h_scale = (float)gs;
  return MS_OK;
}
