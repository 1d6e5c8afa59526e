// Decode / chunked-prefill attention interface.
#pragma once
#include "common.h"

namespace ms {

struct AttnArgs {
  int B, T;                 // sequences, rows per sequence
  int q_dim, kv_dim, hd, n_heads, n_kv, rot;
  int cache_kind, cache_len, clamp;
  float scale;              // 1/sqrt(head_dim)
  // q|k|v rows [B*T][ld]: q at column 0, k at q_dim, v at q_dim + kv_dim
  const float *qkv;
  int ld;
  int apply_rope;
  const float *cos_t, *sin_t;  // [positions][rot/2]
  const int32_t *pos;          // base position per sequence [B]
  float *kc, *vc;              // caches [B][cache_len][kv_dim]
  size_t cache_seq_stride;     // floats between sequences
  int n_chunks;                // chunks of kAttnChunk keys per (sequence, kv head)
  float *part;                 // attn_part_floats(B, n_kv, n_chunks, T, G, hd)
  // combine
  float *out;                  // [B*T][q_dim]
  int write_cache;
  // decode (T == 1): per (sequence, kv head) count of finished chunk blocks;
  // zero on entry, left zero on exit
  unsigned *ctr;
  // prefill (launch_attention_prefill): position of the first row
  int plan_pos;
  // decode: every sequence's position is below pos_bound (0: no bound).  Only
  // the chunks below it are launched, and they load their cached rows before
  // the position arrives.  A position at or past the bound loses its keys
  // beyond the launched chunks: the host must keep the bound.
  int pos_bound;
  int grid_chunks;  // set by the launcher
  // decode partials: cos and sin of the RoPE angles at the row's position,
  // [2][rot / 2] (written before the launch: by the one-row Q|K|V projection
  // or by launch_rope_cur), read at kernel entry instead of the tables
  const float *rope_cur;
};

constexpr int kAttnChunk = 16;
constexpr int kAttnMaxTG = 20;    // T * (n_heads / n_kv) per block
constexpr int kAttnLds = 10240;   // floats of q staging
constexpr int kAttnMaxChunks = 512;

// Floats of AttnArgs::part for B sequences of T rows in n_chunks key chunks.
inline size_t attn_part_floats(int B, int n_kv, int n_chunks, int T, int G, int hd) {
  return (size_t)B * n_kv * ((size_t)n_chunks * T * G * (hd + 2) + 4);
}

// Decode at one row per sequence with the merge left to the consumer: one
// block per (32-key chunk, sequence x kv head) writes the chunk's unnormalized
// o = sum_k e^(s_k - m) v_k and (m, l = sum_k e^(s_k - m)) per query head, and
// the block holding the current slot appends the row's k and v to the cache.
// The O projection merges the chunks (AttnSrc in q4.h).  Per sequence, at
// a.part: o [kDecPartMaxChunks][n_heads][hd], then (m, l)
// [kDecPartMaxChunks][n_heads][2].  Needs G <= 4, head dim 256 or 512 and at
// most kDecPartMaxChunks
// launched chunks (dec_part_ok).
constexpr int kDecPartChunk = 32;
constexpr int kDecPartMaxChunks = 64;
inline size_t dec_part_floats(int B, int n_heads, int hd) {
  return (size_t)B * kDecPartMaxChunks * n_heads * (hd + 2);
}
// Chunks a partials launch covers (the host's position bound, else the cache).
int dec_part_chunks(const AttnArgs &a);
bool dec_part_ok(const AttnArgs &a);
// Counters a model keeps for the decode attention (zero between launches):
// k_attn_decode uses one per (sequence, kv head), the merging partials one per
// (sequence, kv head, pair of query heads).
inline size_t attn_ctr_count(int max_seqs, int n_kv) { return (size_t)max_seqs * n_kv * 2; }
// merge = true: the same blocks, the RoPE factors from the tables at each
// sequence's position, and the last block of each (sequence, kv head, pair of
// query heads) merges the chunks into a.out [B][q_dim] (a.ctr: B * n_kv * 2
// counters, zero between launches).
int launch_attention_partials(const AttnArgs &a, hipStream_t st, bool merge = false);
// The partials of a batch, one row of each sequence (RoPE factors from the tables
// at each position), for launch_merge_quant (q4.h).  attn_batch_ok: shapes taken.
bool attn_batch_ok(const AttnArgs &a);
int launch_attention_batch(const AttnArgs &a, hipStream_t st);
int launch_attention_batch_merged(const AttnArgs &a, hipStream_t st);
// Two to four rows of one sequence on a linear cache (attn_rows_ok): the
// chunk scheme of the decode step per row (k_attn_rows), then the chunks
// merged per row and query head into a.out [T][q_dim].  The partials need
// dec_part_floats(T, ...).
bool attn_rows_ok(const AttnArgs &a);
int launch_attention_rows(const AttnArgs &a, hipStream_t st);
// a.rope_cur from the tables at the position of sequence 0 (one block)
int launch_rope_cur(const AttnArgs &a, hipStream_t st);

// T == 1 (decode): one launch; the chunk blocks append the row to the cache and
// the last block of each (sequence, kv head) merges the chunks (needs a.ctr).
// T > 1: scores + chunk softmax + P.V partials, then the merge of the chunks
// with the cache append of the rows (two launches).
int launch_attention(const AttnArgs &a, hipStream_t st);
int attn_check(const AttnArgs &a);

// Prefill attention of T rows of one sequence (B = 1) at positions plan_pos ..
// plan_pos + T - 1 (flash.hip): RoPE, causal attention over the cached keys and
// the rows' own, and the cache append of the rows.  Any number of query heads
// per kv head; a.part and a.pos are not used.  buf: flash_bytes(a) bytes of
// workspace, never more than flash_bytes_max(a) at the same T, whatever the
// position.
struct FlashBuf {
  int base, kbase;        // first row's position; first key of tile 0
  int nkt, n_qt;          // 32-key tiles; tiles of 64 queries per kv head
  int st_tiles, maxs;     // key tiles per split, splits per query tile (1: none)
  int append;             // k_flash_prep appends the rows to the cache
  __bf16 *q, *k, *v;      // operands in three parts, in MFMA fragment order
  int32_t *bad;           // per key tile: k or v holds a value that is not finite
  float *part;            // per split block: o [64][hd], then (max, sum) [64][2]
};
size_t flash_bytes(const AttnArgs &a);
size_t flash_bytes_max(const AttnArgs &a);
int launch_attention_prefill(const AttnArgs &a, void *buf, size_t buf_bytes, hipStream_t st);

}  // namespace ms
