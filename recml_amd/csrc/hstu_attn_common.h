// What the attention kernels of hstu_attn.hip and hstu_f32.hip share: the argument block of a launch, a sequence's
// geometry, and dropout's keep rule.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hstu_attn.h"

namespace hstu {

typedef __bf16 bf16_t;
typedef bf16_t bf16x8 __attribute__((ext_vector_type(8)));
typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Where the blocks of the logits' gradients of one (sequence, head) lie that a backward's kernels hand on: row i's block j at slot
// i * step + shift + j, with step < 0 at i (i + 1) / 2 + j; `per_row` slots are allotted for each row of blocks.
struct DsRows {
  int32_t per_row, step, shift;
};

struct Params {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  int64_t q_sb, q_st, q_sh;
  int64_t k_sb, k_st, k_sh;
  int64_t v_sb, v_st, v_sh;
  int64_t o_sb, o_st, o_sh;
  const int32_t* seq_lens;
  const int32_t* seq_offsets;
  const int32_t* q_seg;
  const int32_t* kv_seg;
  const uint8_t* mask;
  const float* dense_bias;
  const float* pos_tab;
  const float* ts_tab;
  const int64_t* ts;
  const float* pos_scaled;   // workspace: log2(e) * pos_tab, zero-padded (MFMA kernel)
  // workspace of the MFMA kernel's timestamp path: per sequence, 1 when max - min timestamp fits
  // 31 bits; then timestamps minus the sequence minimum as int32, and their (min, max) per 32-key tile
  const int32_t* ts_ok;
  const int32_t* ts_rel;
  const int32_t* ts_range;
  const int4* ts_keyed;      // workspace: the bucket tables [heads][3 KB], see TsKeys
  const void* ws_base;       // start of the workspace (all of the above lie within 4 GB of it)
  const float* q_scale;      // [H] or null: dequantisation scales of fp8 q / k
  const float* k_scale;
  int64_t ts_sb;
  int32_t B, L, Lkv, H, d_qk, d_v;
  int32_t jagged, causal, mask_mode, window;
  int32_t mask_batched, dense_bias_batched, pos_heads, ts_heads;
  int32_t mask_pitch, bias_pitch;   // bytes and floats from one row of the keep-mask and of the dense bias to the next
  int32_t weights_in_parts;         // the matrix-core forward: activated weights as two bf16 parts in the second product
  int32_t ts_nb;
  float ts_bucket_size;
  float alpha, inv_n;
  int32_t n_qtiles;
  // Key-range splitting (MFMA forward; off when split_cap == 0): hstu_prepare, which sees the lengths,
  // shares a query tile with more steps than twice a slot's average load between up to MAX_CHUNKS workgroups,
  // each covering a contiguous part of the keys and leaving its fp32 partial O^T in `partial`; the
  // workgroup that arrives last at the tile's counter sums them and writes the rows.
  int32_t split_cap;         // chunk slots of the partial buffer (per head)
  int32_t n_slots;           // workgroups that run at once per XCD (what the split decision balances for)
  int32_t level_tiles;       // tiles per slot that the work list's end holds by falling work (see hstu_prepare)
  const int32_t* mask_range; // workspace: per (mask batch, query tile) the first 32-key step with a kept pair and one past the last
  int32_t whole_window;      // forward: the position table as the caller gave it, no workspace (WHOLE instances)
  int32_t persist;           // forward: resident workgroups that loop over the work list
  int32_t chain_bound;       // backward: its longest tile is what lasts (picks dK/dV's order of products)
  int32_t no_stream;         // forward: interior steps through the compiler-scheduled block code too (a comparison switch)
  int32_t mask_pres;         // the preparation also fills the dense mask's presence table (the backward asks for it)
  // Dropout on the attention weights: pair (b, h, i, j) is kept when drop_hash(...) >= drop_thr (0: no dropout).
  // The survivors' scale 1 / (1 - p) is folded into inv_n by the host.
  uint32_t drop_thr, drop_key;
  // Timestamp descriptors (matrix-core forward at d = 128; null = none): one 16-bit word per (32-key step, query
  // row), [step][row] with `ts_desc_pitch` rows per step, built by hstu_prepare (ts_desc_block) for every head and layer of
  // a batch; and per (128-row tile, chunk of TS_DESC_CHUNK steps) the first step in which some row needs the per-pair
  // lookup (INT32_MAX: none).
  const uint16_t* ts_desc;
  const int32_t* ts_tquads;
  int32_t ts_desc_pitch;
  int32_t ts_desc_tiles;     // tile slots of ts_tquads
  int32_t ts_desc_chunks;    // entries per tile slot: chunks of TS_DESC_CHUNK steps
  float* partial;            // [chunk slot][head][BM x d_v floats in register order]
  uint32_t* ctr;             // workspace: [0, 8) draw counters of the XCDs, [8] workgroups done, then from
                             // CTR_RESERVED on one arrival counter per (chunk slot, head); all zero between launches
  // Work list built on the device by hstu_prepare (MFMA kernel; null = workgroups enumerate every
  // possible (sequence, tile) and most exit): sched[0] = number of items, then from
  // sched[4] on one int4 per (sequence, query tile, chunk) that has work:
  // {b | first chunk slot << 14, qt | chunk << 16 | chunks << 24, first token, stored length}.
  const int32_t* sched;
  // backward pass: gradient of out in, gradients of q, k, v out (layouts of out, q, k, v), and
  // fp32 table gradients that are accumulated into (null = not wanted)
  const void* dout;
  const void *q_pre, *k_pre, *v_pre;   // or null: q = silu(q_pre), ... and dq, dk, dv are gradients of those (matrix-core backward)
  void* dq;
  void* dk;
  void* dv;
  float* dpos;
  float* dts;
  float* dbias;              // gradient of the dense bias, or null
  int32_t dbias_fresh;       // it is written, not added to
  // The logits' gradients between the two kernels of a backward (null: each forms them for itself), see ds_blocks of either file: bytes
  // from one head's blocks to the next, and where in it a block lies.
  unsigned char* ds;
  int64_t ds_head;
  DsRows ds_rows;
  int64_t items_max;         // capacity of the list (sizes the grid)
};

// Per-sequence geometry shared by both kernels.
struct Seq {
  int n_q;        // query rows that produce output
  int n_kv;       // keys that may be attended
  int rows;       // rows of the output tile space (L, or n_b when jagged)
  int64_t tok0;   // first token of the sequence in the token axis
  int64_t bq, bk, bv, bo;  // element offsets of (token 0, head h)
  int64_t ts0;    // element offset of timestamp 0
  int n_ts;       // timestamps addressable for this sequence
};

// o0: first token (jagged layout); nraw: the sequence's length as stored (offset difference or
// seq_lens entry; ignored for the padded layout without a length mask).
__device__ __forceinline__ Seq seq_from(const Params& p, int b, int h, int o0, int nraw) {
  Seq s;
  if (p.jagged) {
    int n = nraw;
    n = n < 0 ? 0 : (n > p.L ? p.L : n);
    s.n_q = n; s.n_kv = n; s.rows = n; s.tok0 = o0;
    s.bq = (int64_t)o0 * p.q_st + (int64_t)h * p.q_sh;
    s.bk = (int64_t)o0 * p.k_st + (int64_t)h * p.k_sh;
    s.bv = (int64_t)o0 * p.v_st + (int64_t)h * p.v_sh;
    s.bo = (int64_t)o0 * p.o_st + (int64_t)h * p.o_sh;
  } else {
    int nq = p.L, nk = p.Lkv;
    if (p.mask_mode == HSTU_MASK_LENGTH) {
      int n = nraw;
      n = n < 0 ? 0 : n;
      nq = n < p.L ? n : p.L;
      nk = n < p.Lkv ? n : p.Lkv;
    }
    s.n_q = nq; s.n_kv = nk; s.rows = p.L; s.tok0 = 0;
    s.bq = (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
    s.bk = (int64_t)b * p.k_sb + (int64_t)h * p.k_sh;
    s.bv = (int64_t)b * p.v_sb + (int64_t)h * p.v_sh;
    s.bo = (int64_t)b * p.o_sb + (int64_t)h * p.o_sh;
  }
  if (p.ts_sb != 0) { s.ts0 = (int64_t)b * p.ts_sb; s.n_ts = p.L; }
  else              { s.ts0 = s.tok0;               s.n_ts = s.n_kv; }
  return s;
}

__device__ __forceinline__ void seq_raw(const Params& p, int b, int& o0, int& nraw) {
  o0 = 0;
  nraw = p.L;
  if (p.jagged) {
    o0 = p.seq_offsets[b];
    nraw = p.seq_offsets[b + 1] - o0;
  } else if (p.mask_mode == HSTU_MASK_LENGTH) {
    nraw = p.seq_lens[b];
  }
}

__device__ __forceinline__ Seq seq_info(const Params& p, int b, int h) {
  int o0, nraw;
  seq_raw(p, b, o0, nraw);
  return seq_from(p, b, h, o0, nraw);
}

__device__ __forceinline__ float ldf(const float* p) { return *p; }
__device__ __forceinline__ float ldf(const bf16_t* p) { return (float)*p; }
__device__ __forceinline__ void stf(float* p, float x) { *p = x; }
__device__ __forceinline__ void stf(bf16_t* p, float x) { *p = (bf16_t)x; }

constexpr float LOG2E = 1.4426950408889634f;

// Dropout's keep rule: a counter-based hash of (seed, b, h, i, j), the same on the host, in every kernel and in
// the CPU oracle.  drop_seed_key folds the 64-bit seed (host, once per call), drop_bh_key the sequence and the
// head (once per work item), drop_keep the pair: two multiply-add steps on the indices, of which a kernel hoists
// the one that is fixed for its lane, then drop_keep_mixed.
__host__ __device__ inline uint32_t drop_seed_key(uint64_t seed) {
  uint32_t z = (uint32_t)seed ^ 0x9E3779B9u;
  z = (z ^ (z >> 16)) * 0x85EBCA6Bu;
  z ^= (uint32_t)(seed >> 32);
  z = (z ^ (z >> 13)) * 0xC2B2AE35u;
  return z ^ (z >> 16);
}
__host__ __device__ inline uint32_t drop_bh_key(uint32_t key, uint32_t bh) {
  uint32_t z = key + bh * 0x9E3779B1u;
  z = (z ^ (z >> 15)) * 0x2C1B3C6Du;
  return z ^ (z >> 13);
}
constexpr uint32_t DROP_CI = 0x85EBCA77u, DROP_CJ = 0xC2B2AE3Du;
// ij = kbh + i * DROP_CI + j * DROP_CJ (wrapping)
// (two multiplications with one fold of the high half onto the low half between them: the comparison reads the product
// from its top bits down, which depend on every bit of ij; seven instructions per pair with the index step and the select)
__host__ __device__ inline bool drop_keep_mixed(uint32_t ij, uint32_t thr) {
  uint32_t z = ij * 0x2C1B3C6Du;
  z = (z ^ (z >> 16)) * 0x297A2D39u;
  return z >= thr;
}
__host__ __device__ inline bool drop_keep(uint32_t kbh, uint32_t i, uint32_t j, uint32_t thr) {
  return drop_keep_mixed(kbh + i * DROP_CI + j * DROP_CJ, thr);
}

// (hstu_attn.hip) Records a message for hstu_attn_last_error and returns `code`.
__attribute__((visibility("hidden"))) int fail(int code, const char* fmt, ...);

// (hstu_attn.hip) The timestamp bucket law's integer thresholds: thr[b] is the smallest clipped |dt| whose bucket is >= b
// (INT32_MAX when 1e9 does not reach b); returns the bucket of 1e9.
constexpr int LAW_THR_LEN = 256;
__attribute__((visibility("hidden"))) int bucket_thresholds(float bucket_size, const int32_t** thr);

// What the logits' gradients that a backward's kernels hand on may take of its workspace.
constexpr size_t DS_MAX_BYTES = (size_t)4 << 30;
// Their slots where a sequence has up to nq x nk blocks of `size` rows and keys: those on and below the diagonal (triangle), all, or, where
// that is fewer, the band that a window leaves, from ceil(window / size) blocks before the diagonal to as many behind it (causal: to the
// diagonal itself).
inline DsRows ds_row_slots(int64_t nq, int64_t nk, bool triangle, bool causal, int window, int size) {
  DsRows r;
  r.per_row = (int32_t)(triangle ? (nq + 2) / 2 : nk);              // nq (nq + 1) / 2 blocks by its nq rows
  r.step = triangle ? -1 : r.per_row;
  r.shift = 0;
  if (window >= 0) {
    const int64_t reach = ((int64_t)window + size - 1) / size, band = causal ? reach + 1 : 2 * reach + 1;
    if (band < r.per_row) { r.per_row = (int32_t)band; r.step = (int32_t)band - 1; r.shift = (int32_t)reach; }
  }
  return r;
}

// (hstu_f32.hip) fp32 products at d_qk = d_v in {16, 32, 64, 128} (bf16 storage: 16).  Whether a call is theirs, and the launches.
__attribute__((visibility("hidden"))) bool f32_takes(const Params& p, bool bf16, bool backward);
__attribute__((visibility("hidden"))) int f32_launch_fwd(const Params& p, bool bf16, hipStream_t st);
__attribute__((visibility("hidden"))) size_t f32_ds_bytes(const Params& p, int64_t total_tokens, int64_t* per_head, DsRows* in_head);
__attribute__((visibility("hidden"))) int f32_launch_bwd(const Params& p, bool bf16, hipStream_t st);

}  // namespace hstu
