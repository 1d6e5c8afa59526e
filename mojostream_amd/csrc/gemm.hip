// Q4 GEMM for prefill rows (M > 16) on v_mfma_i32_16x16x64_i8.
//
// The A operand: activation rows quantized by launch_quant_rows3 to 22-bit
// fixed point, X = rint(y 2^s) with max |y| 2^s < 2^22 (s per row), in three
// balanced int8 limbs stored as limb planes (plane l: limb l of every row, in
// the MFMA fragment order of the GEMV's limb rows inside each 128-row
// super-tile of K).  An A tile is 16 rows of one limb plane, so the D fragment
// of limb l gives lane j + 16r the limb-l sums of rows 4r .. 4r + 3 at column
// j, and the three limbs of an output meet in one lane.  (The GEMV's four
// limbs, 31-bit fixed point, would cost a third more MFMAs here, where the
// MFMAs set the time; 22 bits keep every row within 2^-23 of its maximum,
// the rounding of an fp32 product.)  The weights enter as the unsigned
// nibbles n straight from the panel layout (a mask per dword), and the zero
// point comes back per row: sum_k X_k (n_k - 8) = sum_k X_k n_k - 8 * xsum,
// with xsum = sum_k X_k from the quantization.  Each limb's dot product is
// exact in int32; the three limbs of an output combine exactly
// (limb_combine3), minus 8 * xsum, and are scaled by 2^-s and the tensor
// scale.
//
// Tiling.  A block of four waves computes 32 RT activation rows (RT A tiles per
// limb and wave) by 2 PW panels; wave (wr, wc) owns RT 16-row tiles of each limb
// and PW panels: 3 RT PW accumulators and 6 RT PW MFMAs per 128-value step of K.
// Both operands of a step (A 12 RT KiB, B one 1 KiB super-tile per panel) go from
// global memory straight into LDS in a ring of two steps (three for the smallest
// tile), two blocks per CU (2 x 80 KiB for RT = 2, PW = 8), so that one block's
// barriers, start and epilogue overlap the other's MFMAs.  A limb rows are stored
// without padding, chunk c of row r at chunk position c ^ a_swz(r), so the rows
// one fragment read touches fall in different bank groups.
//
// What bounds it: at 2048 rows the operand traffic and the instructions between
// the MFMAs.  A loop of the same MFMAs, LDS reads, unpacking and operand loads
// runs at 3.14 POP/s on this card (3.76 without the operand loads, 4.33 MFMAs
// alone; the nominal 5.0 is not reached).  Measured in the trace of a whole prefill
// (E4B, 2048 rows; the one-row-tile kernel with compiler scheduling on the same
// card): Gate|Up 243 us, 2.65 POP/s (271 us); Down 136 (143), sliding Q|K|V 42.6
// (48.5), full Q|K|V 79 (88); 14B class, 1000 rows: Gate|Up 361 (396), Down 188
// (197).  On a slower card Gate|Up takes 263 us, 2.45 POP/s.
//
// Short prompts leave most CUs idle where the matrix is narrow (O, Down: 20
// column tiles): gemm_ksplit splits K over blocks, whose exact int64 sums
// k_gemm_kcombine adds: the same integer, so the result does not depend on the
// split.  Down at 77 rows: 43 -> 20 us with its combine; E4B prefill of 77 tokens
// 5.4 -> 4.25 ms.
//
// EPI_SWIGLU: wave column wc holds the gate panels of PW / 2 column groups (slots
// j < PW / 2) and the up panels of the same groups, so each output's gate and up
// values meet in one lane (swiglu_inplace, kernels.mojo:519-532).
#include <algorithm>

#include "devutil.h"
#include "q4.h"

namespace ms {
namespace {

constexpr int kLimbs = 3;     // limb planes of the A operand

// LDS position of 16-byte chunk c of A limb row r: c ^ a_swz(r).  The rows
// one A fragment read touches are r0 + 0..15; a 16-byte read goes in phases
// of 8 lanes over 32 banks of 4 bytes (128 bytes per phase), so rows
// r .. r + 7 must take 8 different chunk positions (r & 7), and rows r and
// r + 8 of a 16-lane phase a different one again (the bit r >> 3).
__device__ inline int a_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// Panel pi of the GEMM's 1-3 weight segments (concatenated): its weights,
// scale, first output column and whether it exists.  The candidates come in
// as values: a lambda capturing them would keep them in private memory and
// turn the block-uniform selects into an indexed scratch load.
__device__ inline void seg_panel(int pi, int K, const uint8_t *w0, const uint8_t *w1,
                                 const uint8_t *w2, float s0, float s1, float s2, int n0,
                                 int n1, int n2, int c0, int c1, int c2, const uint8_t **w,
                                 float *sc, int *col, bool *ok) {
  const int si = pi < n0 ? 0 : (pi < n0 + n1 ? 1 : 2);
  const int loc = pi - (si == 0 ? 0 : (si == 1 ? n0 : n0 + n1));
  *ok = pi < n0 + n1 + n2;
  const uint8_t *base = si == 0 ? w0 : (si == 1 ? w1 : w2);
  *w = *ok ? base + (size_t)loc * K * 8 : w0;
  *sc = si == 0 ? s0 : (si == 1 ? s1 : s2);
  *col = (si == 0 ? c0 : (si == 1 ? c1 : c2)) + loc * 16;
}

// Exact limb combine of one output, minus the zero-point term z: each limb's
// int32 dot product is below 2^25 in magnitude (K <= 16384, |limb| <= 128,
// nibble <= 15), so d0 + 2^8 d1 + 2^16 d2 - z is an integer below 2^43,
// formed exactly in double by FMAs.
__device__ inline double limb_combine3(int d0, int d1, int d2, double z) {
  return __builtin_fma((double)d2, 65536.0, __builtin_fma((double)d1, 256.0, (double)d0)) - z;
}

constexpr int kGRows = 32;    // activation rows per row tile of a wave pair
constexpr int kGNT = 256;     // threads per block
constexpr int gemm_stage(int rt, int pw) { return kLimbs * kGRows * rt * 128 + 2048 * pw; }
// K steps in LDS: the smallest tile runs where few blocks share a CU and keeps
// one step more in flight
constexpr int gemm_stages(int rt, int pw) { return rt * pw <= 4 ? 3 : 2; }
constexpr int gemm_lds(int rt, int pw) { return gemm_stages(rt, pw) * gemm_stage(rt, pw); }
// Epilogue of a K part (GemmArgs::ksplit): its exact sums, for k_gemm_kcombine
constexpr int EPI_PART = 100;

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

template <int EPI, int RT, int PW>
__global__ __launch_bounds__(kGNT, 2) void k_gemm(GemmArgs g) {
  constexpr int PS = 2 * PW;                 // panel slots per block
  constexpr int BM = kGRows * RT;            // activation rows per block
  constexpr int CG = PS / 2;                 // SwiGLU: column groups per block
  constexpr int CGW = CG / 2;                // SwiGLU: column groups per wave column
  constexpr int kA = kLimbs * BM * 128;      // A bytes of a stage
  constexpr int kStage = gemm_stage(RT, PW), kStages = gemm_stages(RT, PW);
  static_assert(EPI != EPI_SWIGLU || PW % 2 == 0, "gate and up panels of a wave");
  extern __shared__ __align__(16) uint8_t lds[];
  const int M = launder(g.M), K = launder(g.K);
  const int8_t *limbs = launder(g.a.limbs);
  const int32_t *shift = launder(g.a.shift);
  const int64_t *xsum = launder(g.a.xsum);
  const uint8_t *sw0 = launder(g.seg[0].w), *sw1 = launder(g.seg[1].w),
                *sw2 = launder(g.seg[2].w);
  const float ss0 = launder(g.seg[0].scale), ss1 = launder(g.seg[1].scale),
              ss2 = launder(g.seg[2].scale);
  const int nseg = launder(g.nseg);
  const int sn0 = launder(g.seg[0].n_cols) >> 4;
  const int sn1 = nseg > 1 ? launder(g.seg[1].n_cols) >> 4 : 0;
  const int sn2 = nseg > 2 ? launder(g.seg[2].n_cols) >> 4 : 0;
  const int sc0 = launder(g.seg[0].out_col0), sc1 = launder(g.seg[1].out_col0),
            sc2 = launder(g.seg[2].out_col0);
  float *out = launder(g.out);
  const int ldo = launder(g.ldo);
  const float *resid = EPI == EPI_RESID ? launder(g.resid) : nullptr;
  float *out2 = EPI == EPI_RESID ? launder(g.out2) : nullptr;
  float *sw_out = EPI == EPI_SWIGLU ? launder(g.sw_out) : nullptr;
  const int ldo_sw = EPI == EPI_SWIGLU ? launder(g.ldo_sw) : 0;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int wr = wave & 1, wc = wave >> 1;
  const int r0 = blockIdx.y * BM;
  const int KG = K >> 7;

  // panel slot -> weights, scale, first column, valid (block-uniform selects)
  auto slot = [=](int sl, const uint8_t **w, float *sc, int *col, bool *ok) {
    if constexpr (EPI == EPI_SWIGLU) {
      const int half = sl >= CG ? 1 : 0, cp = blockIdx.x * CG + sl - half * CG;
      *ok = cp < sn0;
      *w = (half == 0 ? sw0 : sw1) + (size_t)(*ok ? cp : 0) * K * 8;
      *sc = half == 0 ? ss0 : ss1;
      *col = cp * 16;
    } else {
      seg_panel(blockIdx.x * PS + sl, K, sw0, sw1, sw2, ss0, ss1, ss2, sn0, sn1, sn2, sc0, sc1,
                sc2, w, sc, col, ok);
    }
  };
  // the panel slot of this wave's accumulator column j
  auto wslot = [&](int j) {
    if constexpr (EPI == EPI_SWIGLU) return j < CGW ? CGW * wc + j : CG + CGW * wc + (j - CGW);
    else return PW * wc + j;
  };
  // this wave loads panel slots wave, wave + 4, .. (an invalid slot loads a
  // valid panel, one past the last slot its first one)
  constexpr int kBL = (PS + 3) / 4;  // B loads per wave per step (the most)
  __amdgpu_buffer_rsrc_t bsrc[kBL];
#pragma unroll
  for (int j = 0; j < kBL; ++j) {
    const uint8_t *w;
    float sc;
    int col;
    bool ok;
    slot(wave + 4 * j < PS ? wave + 4 * j : wave, &w, &sc, &col, &ok);
    bsrc[j] = buffer_of(launder(w), K * 8);
  }
  // A: a stage holds limb rows BM l + m (limb l of block row m); this wave
  // fills rows 8 (RT wave + u) .. + 7 of every limb; lane l writes row
  // + l / 8 at chunk position l % 8, which holds chunk (l % 8) ^ a_swz(row) of
  // the row.  Rows past the planes read zeros.
  const int pr = launder(g.a.plane_rows);
  __amdgpu_buffer_rsrc_t asrc[kLimbs];
#pragma unroll
  for (int l = 0; l < kLimbs; ++l)
    asrc[l] = buffer_of(launder(limbs + ((size_t)l * pr + r0) * K), min(pr - r0, BM) * K);
  int aoff[RT];
#pragma unroll
  for (int u = 0; u < RT; ++u) {
    const int row = 8 * (RT * wave + u) + (lane >> 3);
    aoff[u] = row * K + ((lane & 7) ^ a_swz(row)) * 16;
  }
  auto issue = [&](int G, int stg) {
    uint8_t *sa = lds + stg * kStage;
#pragma unroll
    for (int l = 0; l < kLimbs; ++l)
#pragma unroll
      for (int u = 0; u < RT; ++u)
        load_lds16(asrc[l], sa + (BM * l + 8 * (RT * wave + u)) * 128, aoff[u], G * 128);
#pragma unroll
    for (int j = 0; j < kBL; ++j)
      if (4 * j + 3 < PS || wave + 4 * j < PS)
        load_lds16(bsrc[j], sa + kA + (wave + 4 * j) * 1024, lane * 16, G * 1024);
  };

  // acc[l][u][j]: limb l of block rows 16 (RT wr + u) .. + 15, panel slot wslot(j)
  v4i acc[kLimbs][RT][PW];
#pragma unroll
  for (int a = 0; a < kLimbs; ++a)
#pragma unroll
    for (int u = 0; u < RT; ++u)
#pragma unroll
      for (int j = 0; j < PW; ++j) acc[a][u][j] = v4i{0, 0, 0, 0};

  const int li = lane & 15, lg = lane >> 4;
  const int swz = a_swz(li);  // a_swz(row) for every row this lane reads
  const int apos[2] = {(16 * RT * wr + li) * 128 + ((2 * lg) ^ swz) * 16,
                       (16 * RT * wr + li) * 128 + ((2 * lg + 1) ^ swz) * 16};
  // One K step: two halves of 64 values.  The order is written out and held by
  // scheduling barriers: the next A fragment is read before the MFMAs of each,
  // and the second half's weights are unpacked between MFMAs.  (Left to itself
  // the compiler reads each fragment right before its MFMAs and waits for it.)
  auto compute = [&](int stg) {
    const uint8_t *sa = lds + stg * kStage;
    const uint8_t *sb = sa + kA + lane * 16;
    constexpr int NA = kLimbs * RT;  // A fragments per half step
    v4i af[2];
    auto aread = [&](int h, int t) {
      return *reinterpret_cast<const v4i *>(sa + (BM * (t / RT) + 16 * (t % RT)) * 128 + apos[h]);
    };
    if constexpr (RT * PW <= 12) {
      v4i bf[2][PW];
      u32x4 raw[PW];
      auto unpack = [&](int h, int j) {
        const uint32_t d0 = raw[j][2 * h], d1 = raw[j][2 * h + 1];
        bf[h][j] = v4i{(int)(d0 & 0x0F0F0F0Fu), (int)((d0 >> 4) & 0x0F0F0F0Fu),
                       (int)(d1 & 0x0F0F0F0Fu), (int)((d1 >> 4) & 0x0F0F0F0Fu)};
      };
#pragma unroll
      for (int j = 0; j < PW; ++j)
        raw[j] = *reinterpret_cast<const u32x4 *>(sb + wslot(j) * 1024);
      af[0] = aread(0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < PW; ++j) unpack(0, j);
#pragma unroll
      for (int q = 0; q < 2 * NA; ++q) {
        const int h = q / NA, t = q % NA;
        __builtin_amdgcn_sched_barrier(0);
        if (q + 1 < 2 * NA) af[(q + 1) & 1] = aread((q + 1) / NA, (q + 1) % NA);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < PW; ++j) {
          acc[t / RT][t % RT][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
              af[q & 1], bf[h][j], acc[t / RT][t % RT][j], 0, 0, 0);
          // (the second half's words between the first half's MFMAs)
          if (h == 0 && (q * PW + j) % NA == 0) unpack(1, (q * PW + j) / NA);
        }
      }
    } else {
      // 192 accumulators: one half's weights at a time
      v4i bf[PW];
      u32x2 raw[PW];
      auto braw = [&](int h) {
        asm volatile("" ::: "memory");  // (or the halves' reads become one)
#pragma unroll
        for (int j = 0; j < PW; ++j)
          raw[j] = *reinterpret_cast<const u32x2 *>(sb + wslot(j) * 1024 + 8 * h);
      };
      auto unpack = [&](int j) {
        bf[j] = v4i{(int)(raw[j].x & 0x0F0F0F0Fu), (int)((raw[j].x >> 4) & 0x0F0F0F0Fu),
                    (int)(raw[j].y & 0x0F0F0F0Fu), (int)((raw[j].y >> 4) & 0x0F0F0F0Fu)};
      };
      braw(0);
      af[0] = aread(0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < PW; ++j) unpack(j);
#pragma unroll
      for (int q = 0; q < 2 * NA; ++q) {
        const int t = q % NA;
        __builtin_amdgcn_sched_barrier(0);
        if (q == NA - 2) braw(1);
        if (q + 1 < 2 * NA) af[(q + 1) & 1] = aread((q + 1) / NA, (q + 1) % NA);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < PW; ++j) {
          acc[t / RT][t % RT][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
              af[q & 1], bf[j], acc[t / RT][t % RT][j], 0, 0, 0);
          if (q == NA - 1) {
            if (j > 0) unpack(j - 1);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if (q == NA - 1) unpack(PW - 1);
      }
    }
  };

  // K steps of this block: all of them, or part blockIdx.z of ksplit
  const int ks = EPI == EPI_PART ? launder(g.ksplit) : 1;
  const int G0 = (int)((long)KG * blockIdx.z / ks);
  const int NG = (int)((long)KG * (blockIdx.z + 1) / ks) - G0;
  // Ring of kStages K steps: step i + kStages - 1 is issued into the stage that
  // step i - 1 used, once every wave has passed the barrier after computing it.
  // The barrier is a bare s_barrier after this wave's own loads of step i have
  // landed (a __syncthreads would wait for the later steps' too).
  constexpr int kLoads = kLimbs * RT + kBL;  // a wave's loads per step
  static_assert(kStages == 2 || PS % 4 == 0, "a ring of three counts every wave's loads");
  issue(G0, 0);
  if (kStages == 3 && NG > 1) issue(G0 + 1, 1);
  for (int i = 0; i < NG; ++i) {
    if (kStages == 3 && i + 1 < NG)
      __builtin_amdgcn_s_waitcnt(0x0070 | kLoads);  // vmcnt(kLoads) lgkmcnt(0)
    else
      __builtin_amdgcn_s_waitcnt(0x0070);            // vmcnt(0) lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int n = i + kStages - 1;
    if (n < NG) issue(G0 + n, n % kStages);
    compute(i % kStages);
  }

  // ---- epilogue: lane (column jc, row rr of each A tile)
  const int jc = lane & 15, rr = lane >> 4;
  float wsc[PW];
  int col[PW];
  bool pv[PW];
#pragma unroll
  for (int j = 0; j < PW; ++j) {
    const uint8_t *w;
    slot(wslot(j), &w, &wsc[j], &col[j], &pv[j]);
  }
#pragma unroll
  for (int u = 0; u < RT; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // lane j + 16 rr holds rows 16 (RT wr + u) + 4 rr + i of column j
      const int row = r0 + 16 * (RT * wr + u) + 4 * rr + i;
      if (row >= M) continue;
      if constexpr (EPI == EPI_PART) {
        // exact sums d0 + 2^8 d1 + 2^16 d2
        int64_t *kp = launder(g.kpart) + ((size_t)blockIdx.z * M + row) * ldo;
#pragma unroll
        for (int j = 0; j < PW; ++j)
          if (pv[j])
            kp[col[j] + jc] = (int64_t)acc[0][u][j][i] + ((int64_t)acc[1][u][j][i] << 8) +
                              ((int64_t)acc[2][u][j][i] << 16);
        continue;
      }
      const double rsc = (double)ldexpf(1.0f, -ldg<int32_t>(shift + row));
      const double rz = (double)(8 * ldg<long long>(xsum + row));
      auto value = [&](int j) {
        return (float)(limb_combine3(acc[0][u][j][i], acc[1][u][j][i], acc[2][u][j][i], rz) *
                       rsc * (double)wsc[j]);
      };
      if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
        for (int j = 0; j < CGW; ++j) {
          if (!pv[j]) continue;
          const float gt = value(j), up = value(j + CGW);
          sw_out[(size_t)row * ldo_sw + col[j] + jc] = up * gt * (1.0f / (1.0f + expf(-gt)));
        }
      } else {
#pragma unroll
        for (int j = 0; j < PW; ++j) {
          if (!pv[j]) continue;
          const size_t oi = (size_t)row * ldo + col[j] + jc;
          const float x = value(j);
          if constexpr (EPI == EPI_STORE) {
            out[oi] = x;
          } else if constexpr (EPI == EPI_ACCUMULATE) {
            out[oi] += x;
          } else {
            const float y = resid[oi] + x;
            out[oi] = y;
            if (out2) out2[oi] = y;
          }
        }
      }
    }
}

}  // namespace

// Rows of the quantized operand a GEMM reads: rows of whole tiles of 32.
int gemm_row_pad(int M) { return (M + kGRows - 1) / kGRows * kGRows; }

namespace {

// The tiles, and the time of one K step in a full round of blocks (two per CU),
// microseconds, from launches of 32 to 2048 rows on the E4B and 14B matrices.
struct Tile {
  int rt, pw;
  double step;
};
constexpr Tile kTiles[] = {{2, 8, 2.40}, {2, 6, 1.96}, {2, 5, 1.65},
                           {1, 8, 1.35}, {1, 5, 0.88}, {1, 4, 0.80}};
constexpr int kPartTile = 5;  // the tile of a K part

long gemm_slots() { return 2L * (ctx().n_cu > 0 ? ctx().n_cu : 256); }

dim3 tile_grid(const Tile &t, int M, int np, bool swiglu) {
  const int cols = swiglu ? (np / 2 + t.pw - 1) / t.pw : (np + 2 * t.pw - 1) / (2 * t.pw);
  return dim3(cols, (M + kGRows * t.rt - 1) / (kGRows * t.rt));
}

// Time of a K step of `blocks` blocks: the full rounds, and for what is left 0.58
// of a round with at most one block per CU (a lone block's waves wait for their
// own chain), nearly a whole one above.  Down at 1024, 1536 and 2048 rows (256, 384
// and 512 blocks of the 2 x 5 tile) 88, 128, 149 us; 640 blocks of the 1 x 8 tile
// 1.6 rounds, 640 to 960 of the 1 x 4 tile 1.55 to 2.0.
double step_time(const Tile &t, long blocks) {
  const long slots = gemm_slots(), part = blocks % slots;
  return ((double)(blocks / slots) + (part == 0 ? 0.0 : 2 * part <= slots ? 0.58 : 0.96)) *
         t.step;
}

// The tile with the least time by that rule.
const Tile &gemm_pick(int M, int np, bool swiglu, double *step) {
  const Tile *pick = nullptr;
  for (const Tile &t : kTiles) {
    if (swiglu && t.pw % 2) continue;
    const dim3 g = tile_grid(t, M, np, swiglu);
    const double s = step_time(t, (long)g.x * g.y);
    if (!pick || s < *step) {
      pick = &t;
      *step = s;
    }
  }
  return *pick;
}

template <int RT, int PW>
void launch_tile(const GemmArgs &g, dim3 grid, hipStream_t st) {
  const size_t lds = gemm_lds(RT, PW);
#define MS_GEMM(E) hipLaunchKernelGGL((k_gemm<E, RT, PW>), grid, dim3(kGNT), lds, st, g)
  switch (g.epi) {
    case EPI_STORE: MS_GEMM(EPI_STORE); break;
    case EPI_ACCUMULATE: MS_GEMM(EPI_ACCUMULATE); break;
    case EPI_RESID: MS_GEMM(EPI_RESID); break;
    default:
      if constexpr (PW % 2 == 0) MS_GEMM(EPI_SWIGLU);
      break;
  }
#undef MS_GEMM
}

}  // namespace

// The K parts of a split GEMM added and scaled: row `blockIdx.y`, 256
// columns per block.  The int64 sum is the exact integer the unsplit kernel
// forms with limb_combine, so every output equals the unsplit one.
template <int EPI>
__global__ __launch_bounds__(256) void k_gemm_kcombine(GemmArgs g) {
  const int M = g.M, N = g.ldo, ks = g.ksplit;
  const int row = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
  if (c >= N) return;
  long long t = 0;
  for (int z = 0; z < ks; ++z) t += ldg<long long>(g.kpart + ((size_t)z * M + row) * N + c);
  const double z8 = (double)(8 * ldg<long long>(g.a.xsum + row));
  const float sc = ldexpf(1.0f, -ldg<int32_t>(g.a.shift + row));
  const float v = (float)(((double)t - z8) * (double)sc * (double)g.seg[0].scale);
  float *o = g.out + (size_t)row * N + c;
  if constexpr (EPI == EPI_STORE) {
    *o = v;
  } else if constexpr (EPI == EPI_ACCUMULATE) {
    *o += v;
  } else {
    const float x = g.resid[(size_t)row * N + c] + v;
    *o = x;
    if (g.out2) g.out2[(size_t)row * N + c] = x;
  }
}

size_t gemm_part_bytes() {
  // at most two part blocks per CU, each with the int64 sums of one tile
  const Tile &t = kTiles[kPartTile];
  return (size_t)gemm_slots() * kGRows * t.rt * 32 * t.pw * 8;
}

// The number of parts with the least time: a part's K steps, about 2 us for the
// combine's launch, and the partial sums written and read back at 6 TB/s.  Down
// (K = 10240) at 32, 64, 128, 256 rows: 43.2, 44.2, 45.5, 47.1 us in one part;
// 19.5, 21.5, 27.9, 36.1 split in 8, 6, 3 and 3.  O (K = 2048) gains up to 32 rows
// only (14.4 -> 13.3 us; at 128 rows the split would cost 1.5 us).
int gemm_ksplit(int M, int K, int N) {
  if (M <= kGemvMaxM || K % 128 != 0 || N % 16 != 0) return 1;
  const Tile &t = kTiles[kPartTile];
  const dim3 g = tile_grid(t, M, N / 16, false);
  const long blocks = (long)g.x * g.y;
  const int steps = K / 128;
  double best = 0;
  gemm_pick(M, N / 16, false, &best);
  best *= steps;
  int ks = 1;
  for (int k = 2; k <= 8 && 4 * k <= steps && blocks * k <= gemm_slots(); ++k) {
    const double us = (steps + k - 1) / k * step_time(t, blocks * k) + 2.0 +
                      16e-6 * k * (double)M * N / 6.0;
    if (us < best) {
      best = us;
      ks = k;
    }
  }
  return ks;
}

int launch_gemm(const GemmArgs &g, hipStream_t st) {
  MS_CHECK_ARG(g.M >= 1 && g.K >= 128 && g.K % 128 == 0 && g.K <= kQuantMaxK,
               "GEMM: K must be a multiple of 128 in [128, 16384]");
  MS_CHECK_ARG(g.a.limbs && g.a.shift && g.a.xsum, "GEMM: quantized rows missing");
  MS_CHECK_ARG(g.nseg >= 1 && g.nseg <= 3, "GEMM: 1..3 weight segments");
  for (int i = 0; i < g.nseg; ++i)
    MS_CHECK_ARG(g.seg[i].w && g.seg[i].n_cols > 0 && g.seg[i].n_cols % 16 == 0,
                 "GEMM: segment columns must be a positive multiple of 16");
  if (g.epi == EPI_STORE || g.epi == EPI_ACCUMULATE || g.epi == EPI_RESID) {
    MS_CHECK_ARG(g.out && g.ldo > 0, "GEMM: output missing");
    MS_CHECK_ARG(g.epi != EPI_RESID || g.resid, "GEMM: residual missing");
  } else if (g.epi == EPI_SWIGLU) {
    MS_CHECK_ARG(g.nseg == 2 && g.seg[0].n_cols == g.seg[1].n_cols && g.sw_out,
                 "GEMM: SwiGLU needs gate and up of equal width and an output");
  } else {
    return fail(MS_E_INVALID, "GEMM: unsupported epilogue");
  }
  int np = 0;
  for (int i = 0; i < g.nseg; ++i) np += g.seg[i].n_cols / 16;
  const bool swiglu = g.epi == EPI_SWIGLU;
  if (g.ksplit > 1) {
    MS_CHECK_ARG(!swiglu && g.nseg == 1 && g.kpart && g.ldo == g.seg[0].n_cols &&
                     g.ksplit <= g.K / 128,
                 "GEMM: K split needs one segment, a plain epilogue, ldo = N");
    dim3 grid = tile_grid(kTiles[kPartTile], g.M, np, false);
    grid.z = g.ksplit;
    const dim3 cgrid((g.ldo + 255) / 256, g.M);
    hipLaunchKernelGGL((k_gemm<EPI_PART, 1, 4>), grid, dim3(kGNT), gemm_lds(1, 4), st, g);
    if (g.parts_only) {
      MS_HIP_TRY(hipGetLastError());
      return MS_OK;
    }
    if (g.epi == EPI_STORE)
      hipLaunchKernelGGL(k_gemm_kcombine<EPI_STORE>, cgrid, dim3(256), 0, st, g);
    else if (g.epi == EPI_ACCUMULATE)
      hipLaunchKernelGGL(k_gemm_kcombine<EPI_ACCUMULATE>, cgrid, dim3(256), 0, st, g);
    else
      hipLaunchKernelGGL(k_gemm_kcombine<EPI_RESID>, cgrid, dim3(256), 0, st, g);
    MS_HIP_TRY(hipGetLastError());
    return MS_OK;
  }
  double step = 0;
  const Tile &t = gemm_pick(g.M, np, swiglu, &step);
  const dim3 grid = tile_grid(t, g.M, np, swiglu);
  switch (t.rt * 100 + t.pw) {
    case 208: launch_tile<2, 8>(g, grid, st); break;
    case 206: launch_tile<2, 6>(g, grid, st); break;
    case 205: launch_tile<2, 5>(g, grid, st); break;
    case 108: launch_tile<1, 8>(g, grid, st); break;
    case 105: launch_tile<1, 5>(g, grid, st); break;
    default: launch_tile<1, 4>(g, grid, st); break;
  }
  MS_HIP_TRY(hipGetLastError());
  return MS_OK;
}

}  // namespace ms
