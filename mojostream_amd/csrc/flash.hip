// Prefill attention: many rows of one sequence, causal GQA over the cached
// keys and the rows' own (semantics in attention.hip).
//
// Operands in three bf16 parts.  A value is h + m + l, h its rounding to bf16, m that
// of the rest and l what is left: 8 + 8 + 8 bits and two signs hold the 24 bits of a
// fp32 value (of at least 2^-109 or zero; below, to 2^-133), and every part has fp32's
// range, so no exponent is shared between values: a row's result does not depend on
// the size of others in its tile.  A product takes six v_mfma_f32_16x16x32_bf16 (hh, hm,
// mh, hl, mm, lh) with fp32 sums; what is dropped (ml, lm, ll) is below 2^-25 of the
// product and 2^-28 of it in the mean.  On gfx950 one fp32 16x16x4 MFMA takes as
// long as a bf16 16x16x32: six of the latter do the work of eight of the former.
// (Two fp16 parts with an exponent per tile, three MFMAs: 23 bits near the tile's
// maximum and fewer below 2^-15 of it.)
//
//  k_flash_prep   q and k after RoPE, v, and the cached keys the rows attend
//                 to, split and written in MFMA fragment order (lane l of a
//                 fragment owns the 16 bytes at 16 l), so that the flash
//                 kernel copies whole tiles straight into LDS and reads every
//                 fragment without bank conflicts.  Where the rows are the
//                 sequence's first it also appends them to the cache; where
//                 older keys were read k_cache_append does it afterwards (a
//                 circular cache must not lose a key that a block still
//                 reads).
//  k_flash        one block per (64 queries of a kv head, key split).  The
//                 queries of a kv head are numbered row * G + g: any number G
//                 of query heads per kv head fills the MFMA tiles.  Wave w
//                 owns queries 16w .. 16w + 15 with its q in registers and
//                 computes S^T = K Q^T and O^T = V^T P^T: a lane then holds
//                 one query's scores (keys 4 (l / 16) + e of each 16-key
//                 half tile), which are the B operand of the second product
//                 as they are (V^T is stored with the same key order), and the
//                 softmax needs two lane swaps a tile.
//                 A block whose tiles hold a value that is not finite
//                 (k_flash_prep's flags) goes key by key instead.
//  k_flash_merge  log-sum-exp merge of the key splits.
//
// Error against 64 bits (relative 2-norm, normal q, k and v, scores up to 0.3 to 3 times
// sqrt(hd)): 0.6e-7 to 1.2e-6 at 300 to 2048 rows, 0.5e-7 to 2.0e-7 at 17 rows, below
// that of an fp32 MFMA kernel with one running sum in each of 18 cells (1.2e-7 to 1.8e-6,
// 0.6e-7 to 4.6e-7).  The two fp16 parts took two thirds of this kernel's time; 1.0e-7 to
// 1.3e-6 on these inputs, 0.8e-7 to 3.2e-7 at 17 rows, and 1e-5 to 5e-5 in rows or dims
// beside values 2^24 times theirs.
//
// Measured (E4B, 2048 rows; the fp32 kernel on the same card): sliding layer 63 + 16
// (prep) against 124 + 15 us (RoPE and append launches), full layer 257 + 40 + 13 (merge)
// against 471 + 15 + 12 (a slower card: 70 + 17 and 291 + 40 + 13); 14B class, 1000 rows,
// one layer: 85 + 18 us against 5.0 ms of chunk launches.  Bound by the fragment reads of
// one wave per SIMD and by its softmax: the matrix cores are busy 38% of the time at head
// dim 256.  A short prompt by latency (77 rows: 14.7 + 7.1 against 22.5 + 9.5 us).
#include <algorithm>
#include <cmath>

#include "attention.h"
#include "devutil.h"

namespace ms {
namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kQB = 64;   // queries per block: 16 per wave
constexpr int kKT = 32;   // keys per tile
constexpr int kFlashMaxSplits = 32;
constexpr int kFlashMaxBlocks = 512;  // blocks of a split launch
constexpr int kFrag = 3 * 512;        // values of a fragment: three parts of 1 KiB

// First and last key that the row at position pos attends to.
__host__ __device__ inline void key_span(int circular, int clamp, int cache_len, int pos, int *lo,
                                         int *hi) {
  *lo = circular && pos - cache_len + 1 > 0 ? pos - cache_len + 1 : 0;
  *hi = !circular && clamp && pos > cache_len - 1 ? cache_len - 1 : pos;
}

// Key tiles [*t0, *t1] of query tile qt.
__host__ __device__ inline void tile_span(const AttnArgs &a, const FlashBuf &f, int qt, int *t0,
                                          int *t1) {
  const int G = a.n_heads / a.n_kv, circ = a.cache_kind == MS_CACHE_CIRCULAR;
  const int r0 = qt * kQB / G;
  const int r1 = (qt * kQB + kQB - 1) / G < a.T - 1 ? (qt * kQB + kQB - 1) / G : a.T - 1;
  int lo, hi, d;
  key_span(circ, a.clamp, a.cache_len, f.base + r0, &lo, &d);
  key_span(circ, a.clamp, a.cache_len, f.base + r1, &d, &hi);
  *t0 = (lo - f.kbase) / kKT;
  *t1 = (hi - f.kbase) / kKT;
}

__host__ __device__ inline int split_count(const FlashBuf &f, int nt) {
  const int n = (nt + f.st_tiles - 1) / f.st_tiles;
  return f.maxs == 1 ? 1 : (n < f.maxs ? n : f.maxs);
}

// The parts of eight values.  (A value that rounds past the largest bf16 is cut off
// instead; what is not finite has itself and zeros as its parts.)
__device__ inline void split3(const float *x, bf8 &h, bf8 &m, bf8 &l) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const bool fin = fabsf(x[j]) < INFINITY;
    h[j] = (__bf16)x[j];
    if (fin && !(fabsf((float)h[j]) < INFINITY))
      h[j] = (__bf16)__uint_as_float(__float_as_uint(x[j]) & 0xFFFF0000u);
    const float r = fin ? x[j] - (float)h[j] : 0.f;
    m[j] = (__bf16)r;
    l[j] = (__bf16)(r - (float)m[j]);
  }
}
// the parts of x[0..7] to dst, dst + 512 and dst + 1024
__device__ inline void store_split(const float *x, __bf16 *dst) {
  bf8 h, m, l;
  split3(x, h, m, l);
  *reinterpret_cast<bf8 *>(dst) = h;
  *reinterpret_cast<bf8 *>(dst + 512) = m;
  *reinterpret_cast<bf8 *>(dst + 1024) = l;
}

// Dims d0 .. d0 + 7 of a head row at src, after RoPE at position pos where
// `rope` is set (pairs (i, i + half) over the first rot dims;
// kernels.mojo:579-595).
__device__ inline void load_rope8(const AttnArgs &a, const float *src, int d0, bool rope, int pos,
                                  float *x) {
  const int rot = a.apply_rope ? a.rot : 0, half = rot >> 1;
  const bool r = rope && d0 < rot, low = d0 < half;
  const f4 x0 = ldg<f4>(src + d0), x1 = ldg<f4>(src + d0 + 4);
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = j < 4 ? x0[j] : x1[j - 4];
  if (rot == 0) return;
  if (half % 8 == 0) {
    // the eight dims lie in one half of the rotary dims or past them; what is
    // not rotated loads its own values and the first table entries
    const int pd = !r ? d0 : low ? d0 + half : d0 - half;
    const size_t ti = !r ? 0 : (size_t)pos * half + (low ? d0 : d0 - half);
    const f4 y0 = ldg<f4>(src + pd), y1 = ldg<f4>(src + pd + 4);
    const f4 c0 = ldg<f4>(a.cos_t + ti), c1 = ldg<f4>(a.cos_t + ti + 4);
    const f4 s0 = ldg<f4>(a.sin_t + ti), s1 = ldg<f4>(a.sin_t + ti + 4);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float y = j < 4 ? y0[j] : y1[j - 4], c = j < 4 ? c0[j] : c1[j - 4],
                  s = j < 4 ? s0[j] : s1[j - 4];
      const float t = low ? x[j] * c - y * s : y * s + x[j] * c;
      x[j] = r ? t : x[j];
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int d = d0 + j, i = d < half ? d : d - half;
    if (!rope || d >= rot) continue;
    const float y = ldg<float>(src + (d < half ? d + half : i));
    const float c = ldg<float>(a.cos_t + (size_t)pos * half + i);
    const float s = ldg<float>(a.sin_t + (size_t)pos * half + i);
    x[j] = d < half ? x[j] * c - y * s : y * s + x[j] * c;
  }
}

// Blocks 0 .. nkt * n_kv - 1: K and V of one 32-key tile of a kv head; the
// rest: 32 queries of a kv head each.  A thread takes one piece of eight dims
// of a key or query (two at head dim 512) and one of eight keys of a dim of
// V.  Latency and instruction fetch bound: one piece per thread keeps the code
// at a tenth of four pieces', which ran 20 us on 77 rows, all of it cold code.
template <int HD>
constexpr int prep_threads() {
  return HD < 256 ? 4 * HD : 1024;
}
template <int HD>
__global__ __launch_bounds__(prep_threads<HD>()) void k_flash_prep(AttnArgs a, FlashBuf f) {
  constexpr int NT = prep_threads<HD>();
  constexpr int NP = 4 * HD / NT;  // pieces per thread
  constexpr int PK = HD / 8;       // threads per key or query
  constexpr int KS = HD / 32;      // 32-dim MFMA steps
  __shared__ const float *krow[kKT], *vrow[kKT];
  __shared__ int kslot[kKT], kind[kKT];  // kind: 0 no key, 1 cached, 2 one of the rows
  const int tid = threadIdx.x;
  const int G = a.n_heads / a.n_kv;
  int blk = blockIdx.x;
  if (blk >= f.nkt * a.n_kv) {
    // ---- queries
    blk -= f.nkt * a.n_kv;
    const int h = blk % a.n_kv;
    const size_t nq = (size_t)f.n_qt * kQB;
#pragma unroll 1
    for (int i = 0; i < NP; ++i) {
      const int q = blk / a.n_kv * 32 + (tid + NT * i) / PK, d8 = (tid + NT * i) % PK;
      const int row = q / G, head = h * G + q - row * G;
      const bool ok = row < a.T;
      float x[8];
      load_rope8(a, a.qkv + (ok ? (size_t)row * a.ld + head * HD : 0), 8 * d8, ok, f.base + row,
                 x);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = ok ? x[j] : 0.f;
      store_split(x, f.q + ((h * nq + (q & ~15)) * HD / 512 + (d8 >> 2)) * kFrag +
                         ((d8 & 3) * 16 + (q & 15)) * 8);
    }
    return;
  }
  // ---- keys and values.  A key's row lies in the cache before base (a full
  // linear cache holds none past its end), then among the rows.
  const int h = blk % a.n_kv, kt = blk / a.n_kv;
  const size_t hc = (size_t)h * HD;
  if (tid < kKT) {
    const int k = f.kbase + kt * kKT + tid, r = k - f.base;
    const bool circ = a.cache_kind == MS_CACHE_CIRCULAR;
    const int slot = circ ? k % a.cache_len : k;
    const int kd = r >= 0 ? (r < a.T ? 2 : 0) : (slot < a.cache_len ? 1 : 0);
    const float *kr = a.qkv + (kd == 2 ? (size_t)r * a.ld + a.q_dim + hc : 0);
    krow[tid] = kd == 1 ? a.kc + (size_t)slot * a.kv_dim + hc : kr;
    vrow[tid] = kd == 1 ? a.vc + (size_t)slot * a.kv_dim + hc : kd == 2 ? kr + a.kv_dim : kr;
    kind[tid] = kd;
    // write_kv_sliding / write_kv_full (gemma4_e4b.mojo:211-249): a circular
    // cache keeps the last cache_len rows, a full linear one drops the rest
    kslot[tid] = kd == 2 && (circ ? r >= a.T - a.cache_len : slot < a.cache_len) ? slot : -1;
  }
  __syncthreads();
  float x[NP][8], v[NP][8];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    // V piece (dim, lk): keys 4 lk + 0..3 and 16 + 4 lk + 0..3
    const int dim = (tid + NT * i) % HD, lk = (tid + NT * i) / HD;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[i][j] = ldg<float>(vrow[4 * lk + (j & 3) + 4 * (j & 4)] + dim);
    const int kk = (tid + NT * i) / PK, d8 = (tid + NT * i) % PK;
    load_rope8(a, krow[kk], 8 * d8, kind[kk] == 2, f.kbase + kt * kKT + kk, x[i]);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      x[i][j] = kind[kk] ? x[i][j] : 0.f;
      v[i][j] = kind[4 * lk + (j & 3) + 4 * (j & 4)] ? v[i][j] : 0.f;
    }
  }
  int bad = 0;
#pragma unroll
  for (int i = 0; i < NP; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j)
      bad |= !(fabsf(x[i][j]) < INFINITY) || !(fabsf(v[i][j]) < INFINITY);
  bad = __syncthreads_or(bad);
  if (tid == 0) f.bad[h * f.nkt + kt] = bad;
  const size_t tile = ((size_t)h * f.nkt + kt) * HD / 16 * kFrag;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int dim = (tid + NT * i) % HD, lk = (tid + NT * i) / HD;
    const int kk = (tid + NT * i) / PK, d8 = (tid + NT * i) % PK;
    store_split(x[i], f.k + tile + ((kk >> 4) * KS + (d8 >> 2)) * kFrag +
                          ((d8 & 3) * 16 + (kk & 15)) * 8);
    store_split(v[i], f.v + tile + (dim >> 4) * kFrag + (lk * 16 + (dim & 15)) * 8);
    if (!f.append) continue;
    if (kslot[kk] >= 0) {
      float *d = a.kc + (size_t)kslot[kk] * a.kv_dim + hc + 8 * d8;
      *reinterpret_cast<f4 *>(d) = f4{x[i][0], x[i][1], x[i][2], x[i][3]};
      *reinterpret_cast<f4 *>(d + 4) = f4{x[i][4], x[i][5], x[i][6], x[i][7]};
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int s = kslot[4 * lk + (j & 3) + 4 * (j & 4)];
      if (s >= 0) a.vc[(size_t)s * a.kv_dim + hc + dim] = v[i][j];
    }
  }
}

// The rows' k (after RoPE) and v into the cache, once every key was read.
__global__ __launch_bounds__(256) void k_cache_append(AttnArgs a, int base) {
  const int r = blockIdx.x, pos = base + r;
  const bool circ = a.cache_kind == MS_CACHE_CIRCULAR;
  if (circ ? r < a.T - a.cache_len : pos >= a.cache_len) return;
  const size_t cb = (size_t)(circ ? pos % a.cache_len : pos) * a.kv_dim;
  const float *row = a.qkv + (size_t)r * a.ld + a.q_dim;
  for (int c = 8 * threadIdx.x; c < a.kv_dim; c += 8 * 256) {
    const int d = c % a.hd;
    float o[8];
    load_rope8(a, row + (c - d), d, true, pos, o);
    *reinterpret_cast<f4 *>(a.kc + cb + c) = f4{o[0], o[1], o[2], o[3]};
    *reinterpret_cast<f4 *>(a.kc + cb + c + 4) = f4{o[4], o[5], o[6], o[7]};
    const float *v = row + a.kv_dim + c;
    *reinterpret_cast<f4 *>(a.vc + cb + c) = ldg<f4>(v);
    *reinterpret_cast<f4 *>(a.vc + cb + c + 4) = ldg<f4>(v + 4);
  }
}

// Maximum over the lanes l, l ^ 16, l ^ 32, l ^ 48.
__device__ inline float max_rows(float v) {
  unsigned x = __float_as_uint(v);
  auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  x = __float_as_uint(v);
  r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// e^d for d <= 0: d log2(e) in two parts, so that the exponential of a large
// |d| keeps fp32's accuracy.
__device__ inline float exp_neg(float d) {
  constexpr float kL = 0x1.715476p+0f, kLlo = 0x1.4ae0cp-26f, kLn2 = 0x1.62e43p-1f;
  const float t = d * kL;
  const float r = __builtin_fmaf(d, kLlo, __builtin_fmaf(d, kL, -t));
  const float e = __builtin_amdgcn_exp2f(t);
  // (d = -inf, a masked key, would make r a NaN; a NaN d stays one)
  return d < -104.f ? 0.f : __builtin_fmaf(e, r * kLn2, e);
}

// Instruction order of a product phase of `reads` fragment reads feeding `mfmas`
// MFMAs: nine reads ahead, then three per six MFMAs, and `valus` vector instructions
// (the softmax beside the scores) behind each MFMA.  (Left to itself the compiler
// reads each fragment right before its use and waits for it; with one wave per SIMD
// nothing else covers that.)
template <int READS, int MFMAS, int VALUS>
__device__ inline void interleave() {
  constexpr int kMfma = 0x008, kRead = 0x100, kValu = 0x002;
  __builtin_amdgcn_sched_group_barrier(kRead, 9, 0);
#pragma unroll
  for (int i = 9; i < READS; i += 3) {
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
      if (k & 1) __builtin_amdgcn_sched_group_barrier(kRead, 1, 0);
      if (VALUS > 0) __builtin_amdgcn_sched_group_barrier(kValu, VALUS, 0);
    }
  }
  __builtin_amdgcn_sched_group_barrier(kMfma, MFMAS, 0);
}

// Value j of the fragment piece at p, from its parts.
__device__ inline float whole(const __bf16 *p, int j) {
  return ((float)p[j] + (float)p[512 + j]) + (float)p[1024 + j];
}

// The queries of one wave over key tiles t0 .. t1, key by key in fp32: for blocks whose
// tiles hold values that are not finite.  There the products of parts, and those with
// the weights of masked keys (0 NaN), would reach rows that do not attend to the value.
// Lanes take 64 keys for the scores and HD / 64 dims each for the output.  Not tuned: with
// such a value in every key tile a sliding layer of 2048 rows takes 7.5 ms, a full one 33.
template <int HD, class Store>
__device__ inline void flash_plain(const AttnArgs &a, const FlashBuf &f, int h, int q0, int t0,
                                   int t1, int lane, Store store) {
  constexpr int KS = HD / 32, ND = HD / 64;
  const int G = a.n_heads / a.n_kv, circ = a.cache_kind == MS_CACHE_CIRCULAR;
  const size_t nq = (size_t)f.n_qt * kQB, tile = (size_t)HD / 16 * kFrag;
  const __bf16 *kb = f.k + h * f.nkt * tile, *vb = f.v + h * f.nkt * tile;
#pragma unroll 1
  for (int q = q0; q < q0 + 16; ++q) {
    int lo = 1, hi = 0;
    if (q / G < a.T) {
      key_span(circ, a.clamp, a.cache_len, f.base + q / G, &lo, &hi);
      lo = max(lo - f.kbase, t0 * kKT);
      hi = min(hi - f.kbase, t1 * kKT + kKT - 1);
    }
    const __bf16 *qp = f.q + (h * nq + q0) * HD / 512 * kFrag + (q - q0) * 8;
    float m = -INFINITY, l = 0.f, o[ND];
#pragma unroll
    for (int j = 0; j < ND; ++j) o[j] = 0.f;
#pragma unroll 1
    for (int k0 = lo; k0 <= hi; k0 += 64) {
      const bool on = k0 + lane <= hi;
      const int k = on ? k0 + lane : hi, kk = k % kKT;
      const __bf16 *kp = kb + k / kKT * tile + (kk >> 4) * KS * kFrag + (kk & 15) * 8;
      float s = 0.f;
#pragma unroll 1
      for (int d8 = 0; d8 < HD / 8; ++d8) {
        const int p = (d8 >> 2) * kFrag + (d8 & 3) * 128;
#pragma unroll
        for (int j = 0; j < 8; ++j) s = __builtin_fmaf(whole(qp + p, j), whole(kp + p, j), s);
      }
      const float x = on ? s * a.scale : -INFINITY;
      float mn = x;
#pragma unroll
      for (int i = 1; i < 64; i <<= 1) mn = fmaxf(mn, __shfl_xor(mn, i, 64));
      mn = fmaxf(m, mn);
      const float safe = mn == -INFINITY ? 0.f : mn;
      const float p = on ? expf(x - safe) : 0.f, c = m == -INFINITY ? 0.f : expf(m - safe);
      float ps = p;
#pragma unroll
      for (int i = 1; i < 64; i <<= 1) ps += __shfl_xor(ps, i, 64);
      l = l * c + ps;
      m = mn;
#pragma unroll
      for (int j = 0; j < ND; ++j) o[j] *= c;
#pragma unroll 1
      for (int u = k0; u <= min(hi, k0 + 63); ++u) {
        const float pu = __shfl(p, u - k0, 64);
        const int uk = u % kKT;
        const __bf16 *vp = vb + u / kKT * tile + ((uk >> 2) & 3) * 128;
#pragma unroll
        for (int j = 0; j < ND; ++j) {
          const int d = lane + 64 * j;
          o[j] = __builtin_fmaf(pu, whole(vp + (d >> 4) * kFrag + (d & 15) * 8,
                                          (uk & 3) + (uk >> 4) * 4), o[j]);
        }
      }
    }
    store(q, m, l, o);
  }
}

// Keys and values go through a ring of three LDS stages of up to 48 KiB: a K or V
// tile (half of one at head dim 512: 16 keys of K, 256 dims of V).  Two stages are
// in flight while one is read.  Head dims up to 256 take them in the order K0, K1, V0,
// K2, V1, .. (AHEAD): the scores of tile t + 1 are computed beside the softmax of
// tile t.
template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(HD <= 128 ? 2 : 1, HD <= 128 ? 2 : 1)))
void k_flash(AttnArgs a, FlashBuf f) {
  constexpr int KS = HD / 32, DT = HD / 16;
  constexpr int TB = HD * 192;         // bytes of a K or V tile
  constexpr bool AHEAD = HD <= 256;
  constexpr int NST = AHEAD ? 1 : 2;   // stages of a tile
  constexpr int SB = TB / NST;         // bytes of a stage
  constexpr int NLD = SB / 4096;       // 1 KiB loads per wave and stage
  constexpr int ND = AHEAD ? 4 : 2;    // 16-dim tiles of O in one go
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int li = lane & 15, lk = lane >> 4;
  const int G = a.n_heads / a.n_kv, circ = a.cache_kind == MS_CACHE_CIRCULAR;
  // block (split, query tile, kv head), the tiles with the most keys first and
  // the heads interleaved: heavy blocks start first, and the round-robin of
  // blocks over the XCDs spreads every kind of block
  const int j = blockIdx.x;
  const int h = j % a.n_kv, qt = f.n_qt - 1 - (j / a.n_kv) % f.n_qt, sp = j / (a.n_kv * f.n_qt);
  int t0, t1;
  tile_span(a, f, qt, &t0, &t1);
  const int nsplit = split_count(f, t1 - t0 + 1);
  if (sp >= nsplit) return;
  t0 += sp * f.st_tiles;
  if (sp < nsplit - 1) t1 = t0 + f.st_tiles - 1;
  const int n = t1 - t0 + 1, n_stages = 2 * NST * n;

  const size_t nq = (size_t)f.n_qt * kQB;
  const int qi = qt * kQB + wave * 16 + li, row = qi / G;
  const bool valid = row < a.T;
  int lo, hi;
  key_span(circ, a.clamp, a.cache_len, f.base + row, &lo, &hi);
  lo = valid ? lo - f.kbase : 1;
  hi = valid ? hi - f.kbase : 0;
  int bad = 0;
  for (int t = t0 + lane; t <= t1; t += 64) bad |= ldg<int32_t>(f.bad + h * f.nkt + t);
  bf8 qh[KS], qm[KS], ql[KS];
  {
    const __bf16 *qp = f.q + (h * nq + qt * kQB + wave * 16) * HD / 512 * kFrag + lane * 8;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      qh[s] = ldg<bf8>(qp + s * kFrag);
      qm[s] = ldg<bf8>(qp + s * kFrag + 512);
      ql[s] = ldg<bf8>(qp + s * kFrag + 1024);
    }
  }
  const uint8_t *kg = reinterpret_cast<const uint8_t *>(f.k) + (size_t)h * f.nkt * TB;
  const uint8_t *vg = reinterpret_cast<const uint8_t *>(f.v) + (size_t)h * f.nkt * TB;
  // this wave's NLD kilobytes of stage i, if there is one, into a slot of the ring
  const int voff = wave * (NLD * 1024) + lane * 16;
  auto issue = [&](int i, int slot) {
    if (i >= n_stages) return;
    int t, half = 0;
    bool is_v;
    if constexpr (AHEAD) {
      t = (i - 1) >> 1;
      is_v = i > 0 && (t == n - 1 || !(i & 1));
      t += is_v ? 0 : 1;  // (stage 0: K of tile 0)
    } else {
      t = i >> 2;
      is_v = i & 2;
      half = i & 1;
    }
    const int src = (t0 + t) * TB + half * SB;
    const __amdgpu_buffer_rsrc_t r = buffer_of(is_v ? vg : kg, f.nkt * TB);
    uint8_t *dst = lds + slot * SB + wave * NLD * 1024;
#pragma unroll
    for (int u = 0; u < NLD; ++u) load_lds16(r, dst + u * 1024, voff, src + u * 1024);
  };
  // Stage `stage` (in ring slot `slot`) becomes readable; stage + 2 goes into the
  // slot of stage - 1: the barrier comes after this wave's loads of `stage` (those
  // of stage + 1 may be in flight) and after its reads of stage - 1.
  int stage = -1, slot = 2;
  auto next = [&]() {
    ++stage;
    slot = slot == 2 ? 0 : slot + 1;
    asm volatile("" ::: "memory");
    if (stage + 1 < n_stages)
      __builtin_amdgcn_s_waitcnt(0x0070 | (NLD & 15) | ((NLD >> 4) << 14));
    else
      __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(stage + 2, slot == 0 ? 2 : slot - 1);
    return (const uint8_t *)(lds + slot * SB + lane * 16);
  };
  // S^T of NU x 16 keys (fragments from kt): keys 4 lk + e of query li.  Sums of the
  // small products apart, added last; no MFMA feeds one of the next two.
  constexpr int NU = 2 / NST;
  auto scores = [&](const uint8_t *kt, f4 *s) {
    f4 x[NU], y[NU], z[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) s[u] = x[u] = y[u] = z[u] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < KS; ++d) {
      bf8 kh[NU], km[NU], kl[NU];
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        kh[u] = *reinterpret_cast<const bf8 *>(kt + (u * KS + d) * 3072);
        km[u] = *reinterpret_cast<const bf8 *>(kt + (u * KS + d) * 3072 + 1024);
        kl[u] = *reinterpret_cast<const bf8 *>(kt + (u * KS + d) * 3072 + 2048);
      }
#define MS_QK(k, q, r)              \
  _Pragma("unroll") for (int u = 0; u < NU; ++u) r[u] = \
      __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[u], q[d], r[u], 0, 0, 0)
      MS_QK(kh, qh, s);
      MS_QK(kh, qm, x);
      MS_QK(km, qh, y);
      MS_QK(kh, ql, z);
      MS_QK(km, qm, x);
      MS_QK(kl, qh, y);
#undef MS_QK
    }
    if constexpr (!AHEAD) interleave<3 * NU * KS, 6 * NU * KS, 0>();
#pragma unroll
    for (int u = 0; u < NU; ++u) s[u] += (x[u] + y[u]) + z[u];
  };
  f4 o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = f4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  // softmax of the scores of tile t against the running maximum: p in its
  // parts, l rescaled; returns the factor of o
  auto softmax = [&](int t, const f4 *s, bf8 &ph, bf8 &pm, bf8 &pl) {
    const int k0 = t * kKT;
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = s[i >> 2][i & 3] * a.scale;
    // (no branch for tiles without a masked key: the next tile's MFMAs run beside this)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = k0 + 16 * (i >> 2) + 4 * lk + (i & 3);
      x[i] = k >= lo && k <= hi ? x[i] : -INFINITY;
    }
    const float mt = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])),
                           fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
    const float mn = fmaxf(m, max_rows(mt));
    const float safe = mn == -INFINITY ? 0.f : mn;
    const float c = exp_neg(m - safe);  // (0 before the first key)
    m = mn;
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = exp_neg(x[i] - safe);
      ps += x[i];
    }
    l = l * c + ps;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      ph[i] = (__bf16)x[i];
      const float r = x[i] - (float)ph[i];
      pm[i] = (__bf16)r;
      pl[i] = (__bf16)(r - (float)pm[i]);
    }
    // (in place: not behind the next barrier, where no MFMAs cover it)
    asm volatile("" : "+v"(ph), "+v"(pm), "+v"(pl), "+v"(l));
    return c;
  };
  // O^T = c O^T + V^T P^T for the dims of a stage, the tile's sum apart (one rounding
  // of o per tile)
  auto pv = [&](const uint8_t *vt, int d0, float c, const bf8 ph, const bf8 pm, const bf8 pl) {
#pragma unroll
    for (int d = 0; d < DT / NST; d += ND) {
      bf8 vh[ND], vm[ND], vl[ND];
      f4 r[ND];
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        vh[i] = *reinterpret_cast<const bf8 *>(vt + (d + i) * 3072);
        vm[i] = *reinterpret_cast<const bf8 *>(vt + (d + i) * 3072 + 1024);
        vl[i] = *reinterpret_cast<const bf8 *>(vt + (d + i) * 3072 + 2048);
        r[i] = f4{0.f, 0.f, 0.f, 0.f};
      }
#define MS_PV(v, p)              \
  _Pragma("unroll") for (int i = 0; i < ND; ++i) r[i] = \
      __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[i], p, r[i], 0, 0, 0)
      MS_PV(vl, ph);
      MS_PV(vm, pm);
      MS_PV(vh, pl);
      MS_PV(vm, ph);
      MS_PV(vh, pm);
      MS_PV(vh, ph);
#undef MS_PV
#pragma unroll
      for (int i = 0; i < ND; ++i) o[d0 + d + i] = o[d0 + d + i] * c + r[i];
    }
    interleave<3 * DT / NST, 6 * DT / NST, 0>();
  };

  float *pb = f.part + (size_t)j * kQB * (HD + 2);
  bf8 ph, pm, pl;
  issue(0, 0);
  issue(1, 1);
  if constexpr (AHEAD) {
    f4 s[2];
    const uint8_t *st = next();
    scores(st, s);
#pragma unroll 1
    for (int t = 0; t < n; ++t) {
      if (t < n - 1) st = next();
      f4 sn[2];
      scores(st, sn);  // past the last tile: not used
      const float c = softmax(t0 + t, s, ph, pm, pl);
      interleave<6 * KS, 12 * KS, 32 / KS>();
      st = next();
      pv(st, 0, c, ph, pm, pl);
      s[0] = sn[0];
      s[1] = sn[1];
    }
  } else {
#pragma unroll 1
    for (int t = 0; t < n; ++t) {
      f4 s[2];
      const uint8_t *st = next();
      scores(st, s);
      st = next();
      scores(st, s + 1);
      const float c = softmax(t0 + t, s, ph, pm, pl);
      st = next();
      pv(st, 0, c, ph, pm, pl);
      st = next();
      pv(st, DT / 2, c, ph, pm, pl);
    }
  }
  if (__any(bad)) {
    // (here, where its registers cost the loops nothing)
    flash_plain<HD>(a, f, h, qt * kQB + wave * 16, t0, t1, lane,
                    [&](int q, float m1, float l1, const float *o1) {
      const int row1 = q / G, ql = q % kQB;
      if (nsplit == 1 && row1 >= a.T) return;
      float *d = nsplit == 1 ? a.out + (size_t)row1 * a.q_dim + (h * G + q - row1 * G) * HD
                             : pb + ql * HD;
      const float w = nsplit == 1 ? 1.0f / l1 : 1.0f;
#pragma unroll
      for (int i = 0; i < HD / 64; ++i) d[lane + 64 * i] = o1[i] * w;
      if (nsplit > 1 && lane == 0) {
        pb[kQB * HD + 2 * ql] = m1;
        pb[kQB * HD + 2 * ql + 1] = l1;
      }
    });
    return;
  }
  // the query's sum over its four lanes
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (nsplit == 1) {
    if (!valid) return;
    const float w = 1.0f / l;
    float *op = a.out + (size_t)row * a.q_dim + (h * G + qi - row * G) * HD + 4 * lk;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      *reinterpret_cast<f4 *>(op + 16 * d) = o[d] * w;
    }
    return;
  }
  // partial of this split: o, then (max, sum), per query
  float *po = pb + (wave * 16 + li) * HD + 4 * lk;
#pragma unroll
  for (int d = 0; d < DT; ++d) *reinterpret_cast<f4 *>(po + 16 * d) = o[d];
  if (lk == 0) {
    float *pm = pb + kQB * HD + (wave * 16 + li) * 2;
    pm[0] = m;
    pm[1] = l;
  }
}

// 16 queries of a query tile whose keys were split: weights e^(m_s - M) / L
// through LDS, then float4 sums over the splits.
template <int HD>
__global__ __launch_bounds__(256) void k_flash_merge(AttnArgs a, FlashBuf f) {
  __shared__ float wsh[kFlashMaxSplits][16];
  const int qt = blockIdx.x >> 2, qs = (blockIdx.x & 3) * 16, h = blockIdx.y;
  const int G = a.n_heads / a.n_kv;
  int t0, t1;
  tile_span(a, f, qt, &t0, &t1);
  const int nsplit = split_count(f, t1 - t0 + 1);
  if (nsplit <= 1) return;
  const size_t rec = (size_t)kQB * (HD + 2);
  const float *pb = f.part + ((size_t)(f.n_qt - 1 - qt) * a.n_kv + h) * rec;
  const size_t ss = (size_t)f.n_qt * a.n_kv * rec;
  const int tid = threadIdx.x;
  if (tid < 16) {
    const float *pm = pb + kQB * HD + (qs + tid) * 2;
    float M = -INFINITY, L = 0.f;
    for (int s = 0; s < nsplit; ++s) M = fmaxf(M, pm[s * ss]);
    for (int s = 0; s < nsplit; ++s) {
      const float w = pm[s * ss] == -INFINITY ? 0.f : expf(pm[s * ss] - M);
      wsh[s][tid] = w;
      L += pm[s * ss + 1] * w;
    }
    const float inv = L > 0.f ? 1.0f / L : 0.f;  // (queries past the last row)
    for (int s = 0; s < nsplit; ++s) wsh[s][tid] *= inv;
  }
  __syncthreads();
#pragma unroll 4
  for (int e = tid; e < 16 * HD / 4; e += 256) {
    const int q = e / (HD / 4), d = 4 * (e % (HD / 4));
    const int qi = qt * kQB + qs + q, row = qi / G;
    const float *po = pb + (qs + q) * HD + d;
    f4 acc = f4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < nsplit; ++s) acc += wsh[s][q] * ldg<f4>(po + s * ss);
    if (row < a.T)
      *reinterpret_cast<f4 *>(a.out + (size_t)row * a.q_dim + (h * G + qi - row * G) * HD + d) =
          acc;
  }
}

// Splits of st key tiles, st = the launch's tiles over the CUs' block slots
// (at least 4), so that the blocks make about one round of the chip; no split
// unless the longest query tile is a third longer than st.
void split_plan(const AttnArgs &a, FlashBuf *f) {
  f->maxs = 1;
  f->st_tiles = 1 << 30;
  long tot = 0, maxw = 0;
  for (int qt = 0; qt < f->n_qt; ++qt) {
    int t0, t1;
    tile_span(a, *f, qt, &t0, &t1);
    tot += t1 - t0 + 1;
    maxw = std::max<long>(maxw, t1 - t0 + 1);
  }
  tot *= a.n_kv;
  const long slots = a.hd <= 128 ? 512 : 256;
  long st = std::max(4L, (tot + slots - 1) / slots);
  if (st * 4 > maxw * 3) return;
  long maxs = std::min<long>((maxw + st - 1) / st, kFlashMaxSplits);
  maxs = std::min<long>(maxs, kFlashMaxBlocks / ((long)f->n_qt * a.n_kv));
  if (maxs <= 1) return;
  st = std::max(st, (maxw + maxs - 1) / maxs);
  f->maxs = (int)maxs;
  f->st_tiles = (int)st;
}

size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

// Sizes and, with a buffer, pointers of a launch: T rows at position base.
FlashBuf flash_view(const AttnArgs &a, int base, void *buf, size_t *bytes) {
  FlashBuf f{};
  const int G = a.n_heads / a.n_kv, circ = a.cache_kind == MS_CACHE_CIRCULAR;
  int lo, hi, d;
  key_span(circ, a.clamp, a.cache_len, base, &lo, &d);
  key_span(circ, a.clamp, a.cache_len, base + a.T - 1, &d, &hi);
  f.base = base;
  f.kbase = lo & ~(kKT - 1);
  f.nkt = (hi - f.kbase) / kKT + 1;
  f.n_qt = (a.T * G + kQB - 1) / kQB;
  split_plan(a, &f);
  const size_t nq = (size_t)a.n_kv * f.n_qt * kQB, nk = (size_t)a.n_kv * f.nkt * kKT;
  uint8_t *p = static_cast<uint8_t *>(buf);
  size_t off = 0;
  auto take = [&](size_t b) {
    uint8_t *r = p + off;
    off += up256(b);
    return r;
  };
  f.q = reinterpret_cast<__bf16 *>(take(nq * a.hd * 6));
  f.k = reinterpret_cast<__bf16 *>(take(nk * a.hd * 6));
  f.v = reinterpret_cast<__bf16 *>(take(nk * a.hd * 6));
  f.bad = reinterpret_cast<int32_t *>(take((size_t)a.n_kv * f.nkt * 4));
  f.part = reinterpret_cast<float *>(
      take(f.maxs > 1 ? (size_t)f.maxs * f.n_qt * a.n_kv * kQB * (a.hd + 2) * 4 : 0));
  *bytes = off;
  return f;
}

template <int HD>
void launch_hd(const AttnArgs &a, const FlashBuf &f, hipStream_t st) {
  constexpr int lds = 3 * 192 * (HD <= 256 ? HD : HD / 2);
  hipLaunchKernelGGL(k_flash_prep<HD>, dim3((f.nkt + 2 * f.n_qt) * a.n_kv),
                     dim3(prep_threads<HD>()), 0, st, a, f);
  hipLaunchKernelGGL(k_flash<HD>, dim3(f.maxs * f.n_qt * a.n_kv), dim3(256), lds, st, a, f);
  if (f.maxs > 1)
    hipLaunchKernelGGL(k_flash_merge<HD>, dim3(f.n_qt * 4, a.n_kv), dim3(256), 0, st, a, f);
}

}  // namespace

size_t flash_bytes(const AttnArgs &a) {
  size_t b = 0;
  (void)flash_view(a, a.plan_pos, nullptr, &b);
  return b;
}

size_t flash_bytes_max(const AttnArgs &a) {
  // the most keys: a full window or cache before the rows; the most blocks
  const int G = a.n_heads / a.n_kv;
  const size_t nq = (size_t)a.n_kv * ((a.T * G + kQB - 1) / kQB) * kQB;
  const size_t keys = a.cache_kind == MS_CACHE_CIRCULAR ? (size_t)a.cache_len + a.T : a.cache_len;
  const size_t nk = (size_t)a.n_kv * (keys + 2 * kKT);
  return nq * a.hd * 6 + 2 * nk * a.hd * 6 + nk + 8 * 256 +
         (size_t)kFlashMaxBlocks * kQB * (a.hd + 2) * 4;
}

int launch_attention_prefill(const AttnArgs &a, void *buf, size_t buf_bytes, hipStream_t st) {
  if (int rc = attn_check(a)) return rc;
  MS_CHECK_ARG(a.B == 1 && a.plan_pos >= 0 && a.qkv && a.out && a.kc && a.vc && buf,
               "prefill attention: one sequence, its position and its buffers");
  MS_CHECK_ARG(a.ld % 4 == 0 && (!a.apply_rope || (a.cos_t && a.sin_t)),
               "prefill attention: row stride or RoPE tables");
  size_t need = 0;
  FlashBuf f = flash_view(a, a.plan_pos, buf, &need);
  MS_CHECK_ARG(buf_bytes >= need, "prefill attention: workspace too small");
  f.append = a.write_cache && f.kbase == 0 && f.base == 0;
  switch (a.hd) {
    case 64: launch_hd<64>(a, f, st); break;
    case 128: launch_hd<128>(a, f, st); break;
    case 256: launch_hd<256>(a, f, st); break;
    default: launch_hd<512>(a, f, st); break;
  }
  if (a.write_cache && !f.append)
    hipLaunchKernelGGL(k_cache_append, dim3(a.T), dim3(256), 0, st, a, f.base);
  MS_HIP_TRY(hipGetLastError());
  return MS_OK;
}

}  // namespace ms
