// HSTU attention with fp32 products, forward and backward, at d_qk = d_v in {16, 32, 64, 128}: the kernels of fp32 callers
// (Keras' default dtype, the reference operator's own test recipe) and of bf16 models with head dims of 16.
//
//   hstu_f32_fwd   64 query rows per workgroup, 16 per wave; keys streamed:  S^T = K Q^T, pointwise, O^T += V^T P^T
//   hstu_f32_dq    the same rows:  S^T = K Q^T, dP^T = V dO^T, pointwise, dQ^T += K^T dS^T; the gradients of the bias tables
//                  and of the dense bias
//   hstu_f32_dq_ds the same from the blocks of dS that hstu_f32_dkv has left:  dQ^T += K^T dS^T
//   hstu_f32_dkv   64 keys per workgroup, 16 per wave; query rows streamed:  S = Q K^T, dP = dO V^T, pointwise,
//                  dV^T += dO^T P, dK^T += Q^T dS
//
// What bounds them is the fp32 matrix rate (157 TFLOP/s: 32 cycles per v_mfma_f32_16x16x4_f32).  The layout serves that:
//   * A wave's own rows (Q, dO or K, V) stay in registers as the B operand of the products over the channels; the streamed
//     rows come from LDS as the A operand.  The order of a dot product's terms is free, so k-slot l / 16 of product 4 s + e
//     takes channel 16 s + 4 (l / 16) + e: one 16-byte read feeds four products.
//   * The result of S^T is already the B operand of the product over the keys: register r of lane l holds key 4 (l / 16) + r,
//     which is k-slot l / 16 of the r-th product.  Its A operand is read across the channels; the channel that a row of an
//     output block stands for is free as well, so block 4 X + e takes channels 64 X + 4 i + e: again 16 bytes per four
//     products, and 16-byte stores of the result.
//   * One image of a tile serves both kinds of read.  The 16-byte pieces of a row are permuted by an exclusive-or with the
//     row, which spreads sixteen rows over all banks; the permutation is applied to the source address, so tiles come
//     straight from global memory (global_load_lds) into one of two buffers while the other is computed on: one barrier
//     per step and no registers on the way.
//   * 16 x 16 blocks instead of 32 x 32: causal, window, segment and mask blocks that keep nothing are left out one by one
//     (they keep half the pairs of a packed batch with segment ids), and a wave has 110 - 170 registers, so that 2 - 4 waves
//     per SIMD hide the pointwise part and the barriers.
#include "hstu_attn_common.h"

#include <string.h>

#include <type_traits>

using namespace hstu;

namespace {

constexpr int TILE = 64;         // query rows (keys) of a workgroup
constexpr int WROWS = 16;        // of a wave
constexpr int TAB_MAX_L = 6144;  // table instances: the position gradient's sums of one tile live in LDS
constexpr float LN2 = 0.6931471805599453f;

struct TsThr { int32_t thr[LAW_THR_LEN]; float per_log2; int32_t top; };   // thresholds; ln 2 / bucket size; the last bucket
struct Nothing { int32_t unused; };
template <bool TAB> using TabArg = typename std::conditional<TAB, TsThr, Nothing>::type;

template <int D>
struct Shape {
  static constexpr int CPR = D / 4;                      // 16-byte pieces of a row
  static constexpr int KG = D >= 128 ? 1 : 2;            // groups of 16 streamed rows per step
  static constexpr int KT = 16 * KG;
  static constexpr int NS = D / 16;                      // 16-byte reads of a row per lane; output blocks of 16 channels
  static constexpr int VEC = NS >= 4 ? 4 : NS;           // output blocks that one read across the channels feeds
  static constexpr int NX = NS / VEC;
  static constexpr int TILE_F = KT * D;                  // floats of a tile
  static constexpr int PIECES = 2 * KT * CPR / 64;       // 1 KB pieces of both tiles of a step
  static constexpr int PPW = PIECES / 4;                 // of a wave
  static constexpr int LDS_F = 4 * TILE_F;               // two buffers of two tiles
  static_assert(PIECES % 4 == 0 && PPW >= 1, "whole pieces per wave");
  // Rows per sweep of the banks (256 bytes), and the row's permutation of its pieces.  A 16-byte read is served in groups of
  // lanes {0 - 3, 12 - 15, 20 - 27}, {4 - 11, 16 - 19, 28 - 31} and the same of the upper half: the permutation of rows r and
  // r + 4 (lanes 0 - 15 and 16 - 31 of a read across the channels) must map {0 - 3, 12 - 15} to itself, so row bits 3:2 go
  // 0, 3, 1, 2 (with the plain row the reads across the channels took four more cycles each).
  static constexpr int RPB = CPR >= 16 ? 1 : 16 / CPR;
  static __device__ constexpr int swz(int row) {
    return CPR >= 16 ? (row & 3) | ((row & 4) << 1) | (((row ^ (row >> 1)) & 4)) : (row / RPB) & (CPR - 1);
  }
};

typedef __attribute__((address_space(3))) float* lds_f;
__device__ __forceinline__ void lds_add(float* p, float x) {
  __hip_atomic_fetch_add((lds_f)p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// 64 lanes x 16 bytes from src(lane) to LDS bytes [dst + 16 lane, + 16).  Inline assembly: the compiler neither waits for
// the load nor guards LDS reads against it; the step loop does both (HSTU_F32_WAIT, barrier).
__device__ __forceinline__ void dma16(const void* src, uint32_t lds_dst) {
  const uint32_t base = __builtin_amdgcn_readfirstlane(lds_dst);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(base), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ float4 load4(const float* p) { return *(const float4*)p; }
__device__ __forceinline__ float4 load4(const bf16_t* p) {
  const uint2 u = *(const uint2*)p;
  return float4{__builtin_bit_cast(float, u.x << 16), __builtin_bit_cast(float, u.x & 0xffff0000u),
                __builtin_bit_cast(float, u.y << 16), __builtin_bit_cast(float, u.y & 0xffff0000u)};
}
__device__ __forceinline__ void store4(float* p, float4 v) { *(float4*)p = v; }
__device__ __forceinline__ void store4(bf16_t* p, float4 v) {
  typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));
  *(bf16x4*)p = bf16x4{(bf16_t)v.x, (bf16_t)v.y, (bf16_t)v.z, (bf16_t)v.w};
}

// The two tiles of a step: rows r0 .. of a and b (at most nrows of each), brought by the wave's share of 1 KB pieces.
template <typename T, int D>
struct Tiles {
  using S = Shape<D>;
  static constexpr bool DIRECT = sizeof(T) == 4;
  const T* a;
  const T* b;
  int st_a, st_b;         // bytes from a row to the next (the dispatch keeps them below 2^31)
  int nrows, w, lane;
  float* lds;
  __device__ __forceinline__ void piece(int i, int& row, int& src_c, bool& second, int& lin) const {
    const int pi = w + 4 * i;
    second = pi >= S::PIECES / 2;
    lin = (second ? pi - S::PIECES / 2 : pi) * 64 + lane;
    row = lin / S::CPR;
    src_c = (lin % S::CPR) ^ S::swz(row);
  }
  __device__ __forceinline__ void fetch(int r0, int buf) const {
#pragma unroll
    for (int i = 0; i < S::PPW; ++i) {
      int row, c, lin;
      bool second;
      piece(i, row, c, second, lin);
      int j = r0 + row;
      j = j < nrows ? j : nrows - 1;          // (rows past the end repeat the last one: their pairs are dropped)
      const T* src = (const T*)((const char*)(second ? b : a) + ((int64_t)j * (second ? st_b : st_a) + (int)sizeof(T) * 4 * c));
      float* dst = lds + (2 * buf + (second ? 1 : 0)) * S::TILE_F;
      if constexpr (DIRECT) {
        dma16(src, (uint32_t)(uintptr_t)(dst + (lin - lane) * 4));
      } else {
        *(float4*)(dst + lin * 4) = load4(src);
      }
    }
  }
  __device__ __forceinline__ const float* tile(int buf, int which) const { return lds + (2 * buf + which) * S::TILE_F; }
};

// A B^T over the channels for 16 streamed rows (rows r0 .. r0 + 15 of the tile) and the wave's own (frag).  Two chains of
// products: one alone waits for its own results.
template <int D>
__device__ __forceinline__ floatx4 dot_rows(const float* tile, int row, int g, const float4 (&frag)[D / 16]) {
  using S = Shape<D>;
  const float* base = tile + row * D;
  const int sw = S::swz(row);
  floatx4 even = {0.f, 0.f, 0.f, 0.f}, odd = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < S::NS; ++s) {
    const float4 a = *(const float4*)(base + 4 * ((4 * s + g) ^ sw));
    even = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, frag[s].x, even, 0, 0, 0);
    odd = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, frag[s].y, odd, 0, 0, 0);
    even = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, frag[s].z, even, 0, 0, 0);
    odd = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, frag[s].w, odd, 0, 0, 0);
  }
  return even + odd;
}
// Two of them side by side, a chain each
template <int D>
__device__ __forceinline__ void dot_rows2(floatx4& x, floatx4& y, const float* tx, const float* ty, int row, int g,
                                          const float4 (&fx)[D / 16], const float4 (&fy)[D / 16]) {
  using S = Shape<D>;
  const int sw = S::swz(row);
  x = y = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < S::NS; ++s) {
    const int at = row * D + 4 * ((4 * s + g) ^ sw);
    const float4 a = *(const float4*)(tx + at), c = *(const float4*)(ty + at);
    x = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, fx[s].x, x, 0, 0, 0);
    y = __builtin_amdgcn_mfma_f32_16x16x4f32(c.x, fy[s].x, y, 0, 0, 0);
    x = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, fx[s].y, x, 0, 0, 0);
    y = __builtin_amdgcn_mfma_f32_16x16x4f32(c.y, fy[s].y, y, 0, 0, 0);
    x = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, fx[s].z, x, 0, 0, 0);
    y = __builtin_amdgcn_mfma_f32_16x16x4f32(c.z, fy[s].z, y, 0, 0, 0);
    x = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, fx[s].w, x, 0, 0, 0);
    y = __builtin_amdgcn_mfma_f32_16x16x4f32(c.w, fy[s].w, y, 0, 0, 0);
  }
}
// x where bit r of keep is set, else 0 (by the bits: a branch per pair otherwise)
__device__ __forceinline__ float kept(float x, uint32_t keep, int r) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & (uint32_t)((int32_t)(keep << (31 - r)) >> 31));
}
// o += A^T X over 16 streamed rows: A read across the channels, X = x[r] for row r0 + 4 g + r
template <int D>
__device__ __forceinline__ void dot_cols(floatx4 (&o)[D / 16], const float* tile, int r0, int m, int g, const floatx4& x) {
  using S = Shape<D>;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = r0 + 4 * g + r;
    const float* base = tile + row * D;
    const int sw = S::swz(row);
#pragma unroll
    for (int X = 0; X < S::NX; ++X) {
      const int ch = 64 * X + S::VEC * m;                          // the lane's VEC neighbouring channels
      const float* p = base + 4 * ((ch >> 2) ^ sw) + (ch & 3);
      float v[S::VEC];
      if constexpr (S::VEC == 4) {
        const float4 t = *(const float4*)p;
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
      } else if constexpr (S::VEC == 2) {
        const float2 t = *(const float2*)p;
        v[0] = t.x; v[1] = t.y;
      } else {
        v[0] = *p;
      }
#pragma unroll
      for (int e = 0; e < S::VEC; ++e)
        o[S::VEC * X + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], x[r], o[S::VEC * X + e], 0, 0, 0);
    }
  }
}
// the lane's row of a result: block VEC X + e, register r is channel 64 X + VEC (4 g + r) + e
template <typename T, int D>
__device__ __forceinline__ void store_row(T* row, const floatx4 (&o)[D / 16], float scale, int g) {
  using S = Shape<D>;
#pragma unroll
  for (int X = 0; X < S::NX; ++X) {
    float v[4 * S::VEC];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int e = 0; e < S::VEC; ++e) v[S::VEC * r + e] = o[S::VEC * X + e][r] * scale;
#pragma unroll
    for (int i = 0; i < S::VEC; ++i)
      store4(row + 64 * X + 4 * S::VEC * g + 4 * i, float4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]});
  }
}

// x * sigmoid's factor by the hardware's exp2 and reciprocal (1 ulp each)
__device__ __forceinline__ float sigmoid(float x) { return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x * LOG2E)); }

// Smallest and largest over the wave, as scalars
template <int CTRL, int ROWS>
__device__ __forceinline__ void minmax_step(int& mn, int& mx) {
  const int on = __builtin_amdgcn_update_dpp(mn, mn, CTRL, ROWS, 0xf, false), ox = __builtin_amdgcn_update_dpp(mx, mx, CTRL, ROWS, 0xf, false);
  mn = mn < on ? mn : on;
  mx = mx > ox ? mx : ox;
}
__device__ __forceinline__ void wave_minmax(int& mn, int& mx) {
  minmax_step<0x111, 0xf>(mn, mx);      // row_shr 1, 2, 4, 8: lane 15 of each row of 16 has its row's
  minmax_step<0x112, 0xf>(mn, mx);
  minmax_step<0x114, 0xf>(mn, mx);
  minmax_step<0x118, 0xf>(mn, mx);
  minmax_step<0x142, 0xa>(mn, mx);      // row_bcast 15, 31: lane 63 has the wave's
  minmax_step<0x143, 0xc>(mn, mx);
  mn = __builtin_amdgcn_readlane(mn, 63);
  mx = __builtin_amdgcn_readlane(mx, 63);
}
// ... of scalars over the workgroup's waves (loop bounds must stay scalar)
__device__ __forceinline__ void block_minmax(int& mn, int& mx, int (*ends)[2], int w, int lane) {
  if (lane == 0) { ends[w][0] = mn; ends[w][1] = mx; }
  __syncthreads();
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    mn = mn < ends[x][0] ? mn : ends[x][0];
    mx = mx > ends[x][1] ? mx : ends[x][1];
  }
  mn = __builtin_amdgcn_readfirstlane(mn);
  mx = __builtin_amdgcn_readfirstlane(mx);
}
// the first and last set bit of a non-empty ballot
__device__ __forceinline__ void ballot_ends(uint64_t hit, int at, int& first, int& last) {
  if (hit) {
    const int f = at + __builtin_ctzll(hit), l = at + 63 - __builtin_clzll(hit);
    first = first < f ? first : f;
    last = last > l ? last : l;
  }
}

// The part [lo, hi) of the streamed positions that can matter to own positions [t0, t0 + 64) under segment ids: from the
// first to the last whose id lies between the tile's smallest and largest.  (Packed batches number their sequences in
// order: each tile then meets its own sequences only.)
__device__ __forceinline__ void segment_range(const int32_t* own, int n_own, const int32_t* other, int t0, int tid, int& lo, int& hi) {
  __shared__ int ends[4][2];
  const int lane = tid & 63;
  int i = t0 + lane;
  i = i < n_own ? i : n_own - 1;
  int mn = own[i], mx = mn;
  wave_minmax(mn, mx);
  int first = 0x7fffffff, last = -1;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll 4
  for (int j0 = lo + 64 * w; j0 < hi; j0 += 256) {
    const int j = j0 + lane, id = other[j < hi ? j : hi - 1];
    ballot_ends(__builtin_amdgcn_ballot_w64(j < hi && id >= mn && id <= mx), j0, first, last);
  }
  block_minmax(first, last, ends, w, lane);
  if (last < 0) { hi = lo; return; }
  lo = first;
  hi = last + 1;
}
// The same under an explicit mask, in groups of 16: the first and last group that keeps a pair.  Sixteen bytes per lane,
// at any alignment (a last piece that would cross the row's end starts earlier and says a little too much).
__device__ __forceinline__ void mask_range_rows(const uint8_t* mb, int pitch, int n_rows, int n_cols, int t0, int tid, int& lo, int& hi) {
  __shared__ int ends[4][2];
  const int lane = tid & 63, w = tid >> 6;
  if (n_cols < 16) return;
  int mn = 0x7fffffff, mx = -1;
  for (int c = (lo >> 4) + lane; 16 * c < hi; c += 64) {
    const int off = 16 * c < n_cols - 16 ? 16 * c : n_cols - 16;
    uint32_t any = 0u;
#pragma unroll 8
    for (int rr = 0; rr < WROWS; ++rr) {
      int r = t0 + WROWS * w + rr;
      r = r < n_rows - 1 ? r : n_rows - 1;
      uint4 v;
      __builtin_memcpy(&v, mb + (int64_t)r * pitch + off, 16);
      any |= v.x | v.y | v.z | v.w;
    }
    if (any) { mn = mn < c ? mn : c; mx = mx > c ? mx : c; }
  }
  wave_minmax(mn, mx);
  block_minmax(mn, mx, ends, w, lane);
  if (mx < 0) { hi = lo; return; }
  lo = 16 * mn > lo ? 16 * mn : lo;
  hi = 16 * mx + 16 < hi ? 16 * mx + 16 : hi;
}
__device__ __forceinline__ void mask_range_cols(const uint8_t* mb, int pitch, int n_cols, int t0, int tid, int& lo, int& hi) {
  __shared__ int ends[4][2];
  const int lane = tid & 63, w = tid >> 6;
  if (n_cols < 16) return;
  int mn = 0x7fffffff, mx = -1;
  // four lanes cover the 64 columns of a row, a wave 16 rows
  int off = t0 + 16 * (lane & 3);
  off = off < n_cols - 16 ? off : n_cols - 16;
#pragma unroll 4
  for (int i = lo + 16 * w + (lane >> 2); i < hi; i += 64) {
    uint4 v;
    __builtin_memcpy(&v, mb + (int64_t)i * pitch + off, 16);
    if (v.x | v.y | v.z | v.w) { mn = mn < i ? mn : i; mx = i; }
  }
  wave_minmax(mn, mx);
  block_minmax(mn, mx, ends, w, lane);
  if (mx < 0) { hi = lo; return; }
  lo = mn;
  hi = mx + 1;
}

// LDS of a table instance: thresholds, the head's bucket values, the workgroup's bucket gradient sums
struct TabLds {
  int32_t thr[LAW_THR_LEN + 1];
  float tab[LAW_THR_LEN];
  float hist[LAW_THR_LEN];
};
// every thread of the workgroup; the caller's next barrier publishes it
__device__ __forceinline__ void tab_setup(const Params& p, const TsThr& ta, TabLds& tl, int h, int tid) {
  tl.thr[tid] = ta.thr[tid];
  if (tid == 0) tl.thr[LAW_THR_LEN] = 0x7fffffff;
  tl.tab[tid] = tid <= ta.top ? p.ts_tab[(int64_t)(p.ts_heads > 1 ? h : 0) * (p.ts_nb + 1) + tid] : 0.f;
  tl.hist[tid] = 0.f;
}
// the bucket of a pair's time difference: the logarithm's guess, settled by the integer thresholds (the guess is within one)
__device__ __forceinline__ int tab_bucket(const TsThr& ta, const TabLds& tl, int64_t tq, int64_t tk) {
  int64_t dt = tq - tk;
  if (dt < 0) dt = -dt;
  const int32_t di = dt < 1 ? 1 : (dt > 1000000000LL ? 1000000000 : (int32_t)dt);
  int bk = (int)(__builtin_amdgcn_logf((float)di) * ta.per_log2);
  bk = bk < LAW_THR_LEN - 1 ? bk : LAW_THR_LEN - 1;
  if (di < tl.thr[bk]) --bk;
  else if (di >= tl.thr[bk + 1]) ++bk;
  bk = bk < 0 ? 0 : bk;
  return bk < ta.top ? bk : ta.top;
}
__device__ __forceinline__ int64_t ts_at(const Params& p, const Seq& s, int i) { return p.ts[s.ts0 + (i < s.n_ts - 1 ? i : s.n_ts - 1)]; }

// Four consecutive bias-table entries for keys j .. j + 3 of row i: indices L - 1 + j - i, clamped (pairs outside are dropped)
__device__ __forceinline__ void pos_row4(const float* tab, int L, int i, int j, float (&v)[4]) {
  const int base = L - 1 + j - i;
  if (base >= 0 && base + 3 <= 2 * L - 2) {
    __builtin_memcpy(v, tab + base, 16);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      int x = base + r;
      x = x < 0 ? 0 : (x > 2 * L - 2 ? 2 * L - 2 : x);
      v[r] = tab[x];
    }
  }
}

// The wave's kept pairs of a 16 x 16 block and their biases, for a lane that holds pairs (i_r, j_r), r < 4.
//   BY_ROW: the query row is the lane's (qi) and the keys are j0 + 4 g + r; else the key is the lane's and the rows stream.
template <bool TAB, bool DEN, bool BY_ROW>
struct Pairs {
  const Params& p;
  const Seq& s;
  int b, h;
  int own;                       // the lane's own position
  int lo, hi;                    // streamed positions the index rules keep for it
  int own_seg;
  bool by_seg;
  uint32_t drop_own;
  int64_t ts_own;
  const float* pos_tab;
  const uint8_t* mask;
  const float* dense;

  __device__ __forceinline__ Pairs(const Params& p_, const Seq& s_, int b_, int h_, int own_) : p(p_), s(s_), b(b_), h(h_), own(own_) {
    const int n_stream = BY_ROW ? s.n_kv : s.n_q, n_own = BY_ROW ? s.n_q : s.n_kv;
    lo = 0;
    hi = n_stream - 1;
    if (p.causal) {
      if (BY_ROW) hi = own < hi ? own : hi;
      else lo = own;
    }
    if (p.window >= 0) {
      hi = own + p.window < hi ? own + p.window : hi;
      lo = own - p.window > lo ? own - p.window : lo;
    }
    if (own >= n_own) hi = -1;
    by_seg = p.mask_mode == HSTU_MASK_SEGMENT;
    own_seg = 0;
    const int oc = own < n_own - 1 ? own : n_own - 1;
    if (by_seg) own_seg = BY_ROW ? p.q_seg[(int64_t)b * p.L + oc] : p.kv_seg[(int64_t)b * p.Lkv + oc];
    drop_own = 0u;
    if (p.drop_thr)
      drop_own = drop_bh_key(p.drop_key, (uint32_t)b * (uint32_t)p.H + (uint32_t)h) + (uint32_t)own * (BY_ROW ? DROP_CI : DROP_CJ);
    if constexpr (TAB) {
      pos_tab = p.pos_tab ? p.pos_tab + (int64_t)(p.pos_heads > 1 ? h : 0) * (2 * p.L - 1) : nullptr;
      ts_own = p.ts_tab ? ts_at(p, s, BY_ROW ? own + 1 : own) : 0;
    }
    if constexpr (DEN) {
      mask = p.mask ? p.mask + (p.mask_batched ? (int64_t)b * p.L * p.mask_pitch : 0) : nullptr;
      dense = p.dense_bias ? p.dense_bias + (p.dense_bias_batched ? (int64_t)b * p.L * p.bias_pitch : 0) : nullptr;
    }
  }

  // What a block's four pairs need from memory, asked for one step ahead (a wait for these would also wait for the tiles on
  // their way): segment ids, mask bytes, dense bias or position-table entries, timestamps.
  struct Raw {
    int32_t seg[4];
    uint32_t word;
    float bias[4];
    int64_t ts[4];
    __device__ __forceinline__ void arrived() {     // (pins the compiler's wait here)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        asm volatile("" : "+v"(seg[r]));
        if constexpr (TAB || DEN) asm volatile("" : "+v"(bias[r]));
        if constexpr (TAB) asm volatile("" : "+v"(ts[r]));
      }
      if constexpr (DEN) asm volatile("" : "+v"(word));
    }
  };
  __device__ __forceinline__ void load(Raw& raw, int c0, int g) const {
    const int x0 = c0 + 4 * g;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      raw.seg[r] = own_seg;
      if constexpr (TAB || DEN) raw.bias[r] = 0.f;
      if constexpr (TAB) raw.ts[r] = 0;
    }
    if constexpr (DEN) raw.word = ~0u;
    if (by_seg) {
      const int32_t* other = BY_ROW ? p.kv_seg + (int64_t)b * p.Lkv : p.q_seg + (int64_t)b * p.L;
      const int n = BY_ROW ? p.Lkv : p.L;
      if (c0 + 16 <= n) {
        __builtin_memcpy(raw.seg, other + x0, 16);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) raw.seg[r] = other[x0 + r < n - 1 ? x0 + r : n - 1];
      }
    }
    if constexpr (DEN) {
      if (mask) {
        if constexpr (BY_ROW) {
          const uint8_t* row = mask + (int64_t)(own < p.L - 1 ? own : p.L - 1) * p.mask_pitch;
          const int base = x0 < p.Lkv - 4 ? x0 : p.Lkv - 4;
          __builtin_memcpy(&raw.word, row + base, 4);
        } else {
          const uint8_t* col = mask + (own < p.Lkv - 1 ? own : p.Lkv - 1);
          uint32_t v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = col[(int64_t)(x0 + r < p.L - 1 ? x0 + r : p.L - 1) * p.mask_pitch];
          raw.word = v[0] | (v[1] << 8) | (v[2] << 16) | (v[3] << 24);
        }
      }
      if (dense) {
        if constexpr (BY_ROW) {
          const float* row = dense + (int64_t)(own < p.L - 1 ? own : p.L - 1) * p.bias_pitch;
          if (c0 + 16 <= p.Lkv) {
            __builtin_memcpy(raw.bias, row + x0, 16);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) raw.bias[r] = row[x0 + r < p.Lkv - 1 ? x0 + r : p.Lkv - 1];
          }
        } else {
          const float* col = dense + (own < p.Lkv - 1 ? own : p.Lkv - 1);
#pragma unroll
          for (int r = 0; r < 4; ++r) raw.bias[r] = col[(int64_t)(x0 + r < p.L - 1 ? x0 + r : p.L - 1) * p.bias_pitch];
        }
      }
    }
    if constexpr (TAB) {
      if (pos_tab) {
        if constexpr (BY_ROW) {
          pos_row4(pos_tab, p.L, own, x0, raw.bias);
        } else {
          // rows x0 + r of key `own`: indices L - 1 + own - x0 - r, the same four entries from the other end
          float v[4];
          pos_row4(pos_tab, p.L, x0 + 3, own, v);
#pragma unroll
          for (int r = 0; r < 4; ++r) raw.bias[r] = v[3 - r];
        }
      }
      if (p.ts_tab) {
#pragma unroll
        for (int r = 0; r < 4; ++r) raw.ts[r] = ts_at(p, s, BY_ROW ? x0 + r : x0 + r + 1);
      }
    }
  }

  // keep[r]: bit r of the result; bias[r] and bucket[r] where there are such
  __device__ __forceinline__ uint32_t operator()(const TabArg<TAB>& ta, const TabLds* tl, const Raw& raw, int c0, int g, float (&bias)[4], int (&bucket)[4]) const {
    const int x0 = c0 + 4 * g;
    uint32_t keep = 0u;
#pragma unroll
    for (int r = 0; r < 4; ++r) keep |= (x0 + r >= lo && x0 + r <= hi) ? 1u << r : 0u;
    if (by_seg) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (raw.seg[r] != own_seg) keep &= ~(1u << r);
    }
    if constexpr (DEN) {
      if (mask) {
        uint32_t word = raw.word;
        if constexpr (BY_ROW) {        // (a word that would cross the row's end was fetched from further left)
          const int base = x0 < p.Lkv - 4 ? x0 : p.Lkv - 4;
          word = x0 - base < 4 ? word >> (8 * (x0 - base)) : 0u;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (((word >> (8 * r)) & 0xffu) == 0u) keep &= ~(1u << r);
      }
    }
    if constexpr (TAB || DEN) {
#pragma unroll
      for (int r = 0; r < 4; ++r) bias[r] = raw.bias[r];
    }
    if constexpr (TAB) {
      if (p.ts_tab) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          bucket[r] = BY_ROW ? tab_bucket(ta, *tl, ts_own, raw.ts[r]) : tab_bucket(ta, *tl, raw.ts[r], ts_own);
          bias[r] += tl->tab[bucket[r]];
        }
      }
    }
    if (p.drop_thr) {
      asm volatile("");        // (a branch, not four hashes and a select for everybody)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (!drop_keep_mixed(drop_own + (uint32_t)(x0 + r) * (BY_ROW ? DROP_CJ : DROP_CI), p.drop_thr)) keep &= ~(1u << r);
    }
    return keep;
  }
};

// The streamed keys [lo, hi) of query rows q0 .. q0 + 63 (lo a multiple of 16)
template <bool DEN>
__device__ __forceinline__ void key_range(const Params& p, const Seq& s, int b, int q0, int tid, int& lo, int& hi) {
  lo = 0;
  hi = s.n_kv;
  if (p.causal && q0 + TILE < hi) hi = q0 + TILE;
  if (p.window >= 0) {
    if (q0 + TILE + p.window < hi) hi = q0 + TILE + p.window;
    if (q0 - p.window > 0) lo = q0 - p.window;
  }
  if (p.mask_mode == HSTU_MASK_SEGMENT && lo < hi)
    segment_range(p.q_seg + (int64_t)b * p.L, p.L, p.kv_seg + (int64_t)b * p.Lkv, q0, tid, lo, hi);
  if constexpr (DEN) {
    if (p.mask && lo < hi)
      mask_range_rows(p.mask + (p.mask_batched ? (int64_t)b * p.L * p.mask_pitch : 0), p.mask_pitch, p.L, p.Lkv, q0, tid, lo, hi);
  }
  lo &= ~15;
}
// The streamed query rows of keys k0 .. k0 + 63
template <bool DEN>
__device__ __forceinline__ void query_range(const Params& p, const Seq& s, int b, int k0, int tid, int& lo, int& hi) {
  lo = p.causal ? k0 : 0;
  hi = s.n_q;
  if (p.window >= 0) {
    if (k0 + TILE + p.window < hi) hi = k0 + TILE + p.window;
    if (k0 - p.window > lo) lo = k0 - p.window;
  }
  if (p.mask_mode == HSTU_MASK_SEGMENT && lo < hi)
    segment_range(p.kv_seg + (int64_t)b * p.Lkv, p.Lkv, p.q_seg + (int64_t)b * p.L, k0, tid, lo, hi);
  if constexpr (DEN) {
    if (p.mask && lo < hi) mask_range_cols(p.mask + (p.mask_batched ? (int64_t)b * p.L * p.mask_pitch : 0), p.mask_pitch, p.Lkv, k0, tid, lo, hi);
  }
  lo &= ~15;
}

// Whether the index rules leave a pair between own positions [o0, o0 + 16) and streamed ones [c0, c0 + 16)
template <bool BY_ROW>
__device__ __forceinline__ bool block_live(const Params& p, int o0, int n_own, int c0, int c_end) {
  if (o0 >= n_own || c0 >= c_end) return false;
  if (p.causal && (BY_ROW ? c0 > o0 + 15 : o0 > c0 + 15)) return false;
  if (p.window >= 0 && (c0 > o0 + 15 + p.window || c0 + 15 + p.window < o0)) return false;
  return true;
}

// Workgroups go to the eight XCDs in turn by their linear index: with the head fastest and the tile slowest every XCD sees
// every tile position and the longest tiles start first.  (A sequence's tiles next to each other, to share their streamed
// rows in L2, was slower: 0.55 instead of 0.49 ms for the forward of the shape below.)
//
// Measured at B = 128, L = 512, H = 8, d = 128 with two packed sequences and padding per row (N(0, 1) inputs, causal):
// forward 1.23 -> 0.49 ms, dq 2.13 -> 0.70, dk / dv 2.88 -> 1.00 against the general kernels, which run every causal step;
// a small call (B = 4, L = 64, H = 2, d = 32) 12.7 -> 5 us.  The products alone are 545 k, 818 k and 1.09 M cycles per SIMD, half of
// that: an fp32 product and a vector instruction do not overlap (3 instructions behind each product cost 8 of its 32 cycles
// with four waves per SIMD), a wave has only eight blocks to spread its prologue over, and waves wait a third of their
// time for tiles and barriers.

template <typename T, int D, bool TAB, bool DEN>
__global__ __launch_bounds__(256, D >= 128 ? 3 : 4) void hstu_f32_fwd(const Params p, const TabArg<TAB> ta) {
  using S = Shape<D>;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ typename std::conditional<TAB, TabLds, Nothing>::type tl;
  const int h = blockIdx.x, b = blockIdx.y, qt = gridDim.z - 1 - blockIdx.z;
  const Seq s = seq_info(p, b, h);
  const int q0 = qt * TILE;
  if (q0 >= s.rows) return;
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = q0 + WROWS * w, qi = r0 + m;
  floatx4 o[S::NS];
#pragma unroll
  for (int x = 0; x < S::NS; ++x) o[x] = floatx4{0.f, 0.f, 0.f, 0.f};
  if (q0 < s.n_q) {
    int lo, hi;
    key_range<DEN>(p, s, b, q0, tid, lo, hi);
    if (lo < hi) {
      const Tiles<T, D> t = {(const T*)p.k + s.bk, (const T*)p.v + s.bv, (int)(p.k_st * sizeof(T)), (int)(p.v_st * sizeof(T)), s.n_kv, w, lane, sm};
      t.fetch(lo, 0);
      float4 qf[S::NS];
      {
        const T* row = (const T*)p.q + s.bq + (int64_t)(qi < s.n_q ? qi : s.n_q - 1) * p.q_st + 4 * g;
#pragma unroll
        for (int x = 0; x < S::NS; ++x) qf[x] = load4(row + 16 * x);
      }
      if constexpr (TAB) {
        if (p.ts_tab) tab_setup(p, ta, tl, h, tid);
      }
      Pairs<TAB, DEN, true> pairs(p, s, b, h, qi);
      const TabLds* tlp = nullptr;
      if constexpr (TAB) tlp = &tl;
      typename decltype(pairs)::Raw raw[S::KG], next[S::KG];
#pragma unroll
      for (int kg = 0; kg < S::KG; ++kg) pairs.load(next[kg], lo + 16 * kg, g);
      int buf = 0;
      for (int kv0 = lo; kv0 < hi; kv0 += S::KT, buf ^= 1) {
        dma_wait();
#pragma unroll
        for (int kg = 0; kg < S::KG; ++kg) { next[kg].arrived(); raw[kg] = next[kg]; }
        __syncthreads();              // the step's tiles are there, and nobody reads the other buffer any more
        if (kv0 + S::KT < hi) {
#pragma unroll
          for (int kg = 0; kg < S::KG; ++kg) pairs.load(next[kg], kv0 + S::KT + 16 * kg, g);
          t.fetch(kv0 + S::KT, buf ^ 1);
        }
#pragma unroll
        for (int kg = 0; kg < S::KG; ++kg) {
          const int c0 = kv0 + 16 * kg;
          if (!block_live<true>(p, r0, s.n_q, c0, hi)) continue;
          float bias[4] = {0.f, 0.f, 0.f, 0.f};
          int bucket[4];
          const uint32_t keep = pairs(ta, tlp, raw[kg], c0, g, bias, bucket);
          if (__builtin_amdgcn_ballot_w64(keep != 0u) == 0) continue;
          floatx4 x = dot_rows<D>(t.tile(buf, 0), 16 * kg + m, g, qf);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float u = p.alpha * x[r];
            if constexpr (TAB || DEN) u += bias[r];
            x[r] = kept(u * sigmoid(u), keep, r);
          }
          dot_cols<D>(o, t.tile(buf, 1), 16 * kg, m, g, x);
        }
      }
    }
  }
  if (qi < s.rows)          // (rows past the sequence: zeros)
    store_row<T, D>((T*)p.out + s.bo + (int64_t)qi * p.o_st, o, qi < s.n_q ? p.inv_n : 0.f, g);
}

// A block's dS to the sums along its diagonals, key - query = 4 g + r - m of lane (m, g): the four registers are brought onto 4 g - m and
// 4 g - m + 16 by shifts within the rows of 16 lanes.  An LDS float atomic takes the CU's LDS 3 cycles a lane: 76 lanes for a block
// instead of 256 (B = 32, L = 512, H = 8, d = 128, position table, both backward kernels: 781 -> 651 us).
template <int CTRL>
__device__ __forceinline__ float lanes_moved(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ void add_diagonals(float* d, const floatx4& x, int m) {
  // register r of lane m is diagonal r - m: lane m - r's where there is one, else that of lane 16 + m - r, 16 further up
  const float near = (x[0] + lanes_moved<0x101>(x[1])) + (lanes_moved<0x102>(x[2]) + lanes_moved<0x103>(x[3]));
  const float far = lanes_moved<0x11f>(x[1]) + lanes_moved<0x11e>(x[2]) + lanes_moved<0x11d>(x[3]);
  lds_add(d, near);
  if (m >= 13) lds_add(d + 16, far);
}

// What a block's dS adds to the gradients of the biases: `diag` is the lane's place among the tile's diagonal sums, dsm LDS for a block of each
// wave.
template <bool TAB, bool DEN>
__device__ __forceinline__ void bias_grads(const Params& p, const TabLds* tl_, float* diag, float* dsm, const floatx4& x, const int (&bucket)[4], bool want_pos,
                                           bool want_ts, int b, int r0, int c0, int m, int g, int w, int lane) {
  TabLds* const tl = const_cast<TabLds*>(tl_);
  if constexpr (TAB) {
    if (want_pos) add_diagonals(diag, x, m);
    if (want_ts) {
      // neighbouring pairs mostly share a bucket: a block with one bucket is summed over the wave first
      const int b0 = __builtin_amdgcn_readfirstlane(bucket[0]);
      const bool same = bucket[0] == b0 && bucket[1] == b0 && bucket[2] == b0 && bucket[3] == b0;
      if (__builtin_amdgcn_ballot_w64(!same) == 0) {
        float sum = (x[0] + x[1]) + (x[2] + x[3]);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 64);
        if (lane == 0) lds_add(tl->hist + b0, sum);
      } else {
        float sum = x[0];
#pragma unroll
        for (int r = 1; r < 4; ++r) {
          if (bucket[r] != bucket[r - 1]) { lds_add(tl->hist + bucket[r - 1], sum); sum = 0.f; }
          sum += x[r];
        }
        lds_add(tl->hist + bucket[3], sum);
      }
    }
  }
  if constexpr (DEN) {
    if (p.dbias) {
      // the block by rows: an instruction then adds four rows of 64 bytes instead of 16 rows of 16
      float* dw = dsm + w * (16 * 17);
#pragma unroll
      for (int r = 0; r < 4; ++r) dw[m * 17 + 4 * g + r] = x[r];
      __builtin_amdgcn_wave_barrier();
      float* dst = p.dbias + (p.dense_bias_batched ? (int64_t)b * p.L * p.Lkv : 0) + (int64_t)r0 * p.Lkv + c0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = dw[(4 * i + g) * 17 + m];
        if (v != 0.f) atomicAdd(dst + (int64_t)(4 * i + g) * p.Lkv + m, v);      // (zero wherever the pair is masked or outside)
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}
// ... and the workgroup's sums to memory
template <bool TAB>
__device__ __forceinline__ void bias_grads_out(const Params& p, const TabArg<TAB>& ta, const TabLds* tl, const float* diag, int n_diag, bool want_pos, bool want_ts,
                                               int h, int lo, int q0, int tid) {
  if constexpr (TAB) {
    if (want_pos || want_ts) {
      __syncthreads();
      if (want_pos) {
        float* dst = p.dpos + (int64_t)(p.pos_heads > 1 ? h : 0) * (2 * p.L - 1);
        const int base = (p.L - 1) + lo - q0 - (TILE - 1);
        for (int e = tid; e < n_diag; e += 256)
          if (diag[e] != 0.f && base + e >= 0 && base + e < 2 * p.L - 1) atomicAdd(dst + base + e, diag[e]);
      }
      if (want_ts && tid <= ta.top && tl->hist[tid] != 0.f)
        atomicAdd(p.dts + (int64_t)(p.ts_heads > 1 ? h : 0) * (p.ts_nb + 1) + tid, tl->hist[tid]);
    }
  }
}

template <typename T, int D, bool TAB, bool DEN>
__global__ __launch_bounds__(256, D >= 128 ? 2 : 3) void hstu_f32_dq(const Params p, const TabArg<TAB> ta) {
  using S = Shape<D>;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ typename std::conditional<TAB, TabLds, Nothing>::type tl;
  __shared__ float dsm[DEN ? 4 * 16 * 17 : 1];          // each wave's block of dS on its way to the dense bias's gradient
  float* const diag = sm + S::LDS_F;                    // position gradient: sums by key - query, from q0 + 63 - lo down
  const int h = blockIdx.x, b = blockIdx.y, qt = gridDim.z - 1 - blockIdx.z;
  const Seq s = seq_info(p, b, h);
  const int q0 = qt * TILE;
  if (q0 >= s.rows) return;
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = q0 + WROWS * w, qi = r0 + m;
  floatx4 o[S::NS];
#pragma unroll
  for (int x = 0; x < S::NS; ++x) o[x] = floatx4{0.f, 0.f, 0.f, 0.f};
  if (q0 < s.n_q) {
    int lo, hi;
    key_range<DEN>(p, s, b, q0, tid, lo, hi);
    if (lo < hi) {
      const Tiles<T, D> t = {(const T*)p.k + s.bk, (const T*)p.v + s.bv, (int)(p.k_st * sizeof(T)), (int)(p.v_st * sizeof(T)), s.n_kv, w, lane, sm};
      t.fetch(lo, 0);
      float4 qf[S::NS], dof[S::NS];
      {
        const int qc = qi < s.n_q ? qi : s.n_q - 1;
        const T* row = (const T*)p.q + s.bq + (int64_t)qc * p.q_st + 4 * g;
        const T* drow = (const T*)p.dout + s.bo + (int64_t)qc * p.o_st + 4 * g;
#pragma unroll
        for (int x = 0; x < S::NS; ++x) { qf[x] = load4(row + 16 * x); dof[x] = load4(drow + 16 * x); }
      }
      const bool want_ts = TAB && p.dts != nullptr && p.ts_tab != nullptr;
      const bool want_pos = TAB && p.dpos != nullptr && p.pos_tab != nullptr;
      const int n_diag = ((hi - lo + 15) & ~15) + TILE;
      if constexpr (TAB) {
        if (p.ts_tab) tab_setup(p, ta, tl, h, tid);
        if (want_pos) for (int e = tid; e < n_diag; e += 256) diag[e] = 0.f;
      }
      Pairs<TAB, DEN, true> pairs(p, s, b, h, qi);
      const TabLds* tlp = nullptr;
      if constexpr (TAB) tlp = &tl;
      typename decltype(pairs)::Raw raw[S::KG], next[S::KG];
#pragma unroll
      for (int kg = 0; kg < S::KG; ++kg) pairs.load(next[kg], lo + 16 * kg, g);
      int buf = 0;
      for (int kv0 = lo; kv0 < hi; kv0 += S::KT, buf ^= 1) {
        dma_wait();
#pragma unroll
        for (int kg = 0; kg < S::KG; ++kg) { next[kg].arrived(); raw[kg] = next[kg]; }
        __syncthreads();              // the step's tiles are there, and nobody reads the other buffer any more
        if (kv0 + S::KT < hi) {
#pragma unroll
          for (int kg = 0; kg < S::KG; ++kg) pairs.load(next[kg], kv0 + S::KT + 16 * kg, g);
          t.fetch(kv0 + S::KT, buf ^ 1);
        }
#pragma unroll
        for (int kg = 0; kg < S::KG; ++kg) {
          const int c0 = kv0 + 16 * kg;
          if (!block_live<true>(p, r0, s.n_q, c0, hi)) continue;
          float bias[4] = {0.f, 0.f, 0.f, 0.f};
          int bucket[4] = {0, 0, 0, 0};
          const uint32_t keep = pairs(ta, tlp, raw[kg], c0, g, bias, bucket);
          if (__builtin_amdgcn_ballot_w64(keep != 0u) == 0) continue;
          floatx4 x, dp;
          dot_rows2<D>(x, dp, t.tile(buf, 0), t.tile(buf, 1), 16 * kg + m, g, qf, dof);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float u = p.alpha * x[r];
            if constexpr (TAB || DEN) u += bias[r];
            const float sg = sigmoid(u);
            x[r] = kept(dp[r] * sg * (1.0f + u * (1.0f - sg)) * p.inv_n, keep, r);
          }
          dot_cols<D>(o, t.tile(buf, 0), 16 * kg, m, g, x);
          bias_grads<TAB, DEN>(p, tlp, diag + (c0 - lo) + 4 * g + (TILE - 1) - (WROWS * w + m), dsm, x, bucket, want_pos, want_ts, b, r0, c0, m, g, w, lane);
        }
      }
      bias_grads_out<TAB>(p, ta, tlp, diag, n_diag, want_pos, want_ts, h, lo, q0, tid);
    }
  }
  if (qi < s.rows)
    store_row<T, D>((T*)p.dq + s.bq + (int64_t)qi * p.q_st, o, qi < s.n_q ? p.alpha : 0.f, g);
}

// dS from hstu_f32_dkv to hstu_f32_dq_ds: blocks of 16 keys x 16 query rows, a key's 16 rows next to each other, 1 KB each, a
// (sequence, head)'s in the slots of DsRows; a sequence's slots begin where `per_row` for each 16 rows before it (an upper bound) end.  A block without a kept pair is neither written nor read.
constexpr int DS_BLOCK = 16 * 16;
__device__ __forceinline__ float* ds_blocks(const Params& p, int b, int h, const Seq& s) {
  const int64_t rows = p.jagged ? (s.tok0 >> 4) + b : (int64_t)b * ((p.L + 15) >> 4);
  return (float*)(p.ds + (int64_t)h * p.ds_head) + rows * p.ds_rows.per_row * DS_BLOCK;
}
__device__ __forceinline__ int64_t ds_block_at(const Params& p, int i, int j) {
  return (int64_t)((p.ds_rows.step < 0 ? i * (i + 1) / 2 : i * p.ds_rows.step) + p.ds_rows.shift + j) * DS_BLOCK;
}

// The rows of hstu_f32_dq with dS read (the bits it would form): one product of three, the bias gradients as there.  Steps of 32 keys: a tile
// of K alone is half of a step's there.  Bound by that product (B = 128,
// L = 512, H = 8, d = 128 with segment ids: 290 us where hstu_f32_dq takes 678, and hstu_f32_dkv as long as without its stores) and below
// d = 128 by the blocks' reads.
template <int D, bool TAB, bool DEN>
__global__ __launch_bounds__(256, D >= 128 && (TAB || DEN) ? 3 : 4) void hstu_f32_dq_ds(const Params p, const TabArg<TAB> ta) {
  using S = Shape<D>;
  constexpr int KT = 32, TILE_F = KT * D, PPW = KT * S::CPR / 64 / 4;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ typename std::conditional<TAB, TabLds, Nothing>::type tl;
  __shared__ float dsm[DEN ? 4 * 16 * 17 : 1];
  float* const diag = sm + 2 * TILE_F;
  const int h = blockIdx.x, b = blockIdx.y, qt = gridDim.z - 1 - blockIdx.z;
  const Seq s = seq_info(p, b, h);
  const int q0 = qt * TILE;
  if (q0 >= s.rows) return;
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = q0 + WROWS * w, qi = r0 + m;
  floatx4 o[S::NS];
#pragma unroll
  for (int x = 0; x < S::NS; ++x) o[x] = floatx4{0.f, 0.f, 0.f, 0.f};
  if (q0 < s.n_q) {
    int lo, hi;
    key_range<DEN>(p, s, b, q0, tid, lo, hi);
    if (lo < hi) {
      const float* const kg_ = (const float*)p.k + s.bk;
      auto fetch = [&](int kv0, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PPW; ++i) {
          const int lin = (w + 4 * i) * 64 + lane, row = lin / S::CPR, c = (lin % S::CPR) ^ S::swz(row);
          int j = kv0 + row;
          j = j < s.n_kv ? j : s.n_kv - 1;          // (rows past the end repeat the last one: their pairs are 0)
          dma16(kg_ + (int64_t)j * p.k_st + 4 * c, (uint32_t)(uintptr_t)(sm + buf * TILE_F + (lin - lane) * 4));
        }
      };
      const float* const dsg = ds_blocks(p, b, h, s) + m;
      const bool want_ts = TAB && p.dts != nullptr && p.ts_tab != nullptr;
      const bool want_pos = TAB && p.dpos != nullptr && p.pos_tab != nullptr;
      const int n_diag = ((hi - lo + 15) & ~15) + TILE;
      if constexpr (TAB) {
        if (p.ts_tab) tab_setup(p, ta, tl, h, tid);
        if (want_pos) for (int e = tid; e < n_diag; e += 256) diag[e] = 0.f;
      }
      Pairs<TAB, DEN, true> pairs(p, s, b, h, qi);
      const TabLds* tlp = nullptr;
      if constexpr (TAB) tlp = &tl;
      if constexpr (TAB) pairs.pos_tab = nullptr;      // (which pairs are kept and in which bucket is all that is asked)
      if constexpr (DEN) pairs.dense = nullptr;
      struct Block { typename Pairs<TAB, DEN, true>::Raw raw; float x[4]; } next[KT / 16];
      auto ask = [&](Block& to, int c0) __attribute__((always_inline)) {
        pairs.load(to.raw, c0, g);
#pragma unroll
        for (int r = 0; r < 4; ++r) to.x[r] = 0.f;
        if (block_live<true>(p, r0, s.n_q, c0, hi)) {
          const float* const at = dsg + ds_block_at(p, r0 >> 4, c0 >> 4) + 64 * g;
#pragma unroll
          for (int r = 0; r < 4; ++r) to.x[r] = at[16 * r];
        }
      };
      fetch(lo, 0);
#pragma unroll
      for (int kg = 0; kg < KT / 16; ++kg) ask(next[kg], lo + 16 * kg);
      int buf = 0;
      for (int kv0 = lo; kv0 < hi; kv0 += KT, buf ^= 1) {
        Block now[KT / 16];
        dma_wait();
#pragma unroll
        for (int kg = 0; kg < KT / 16; ++kg) {
          next[kg].raw.arrived();
#pragma unroll
          for (int r = 0; r < 4; ++r) asm volatile("" : "+v"(next[kg].x[r]));
          now[kg] = next[kg];
        }
        __syncthreads();              // the step's tile is there, and nobody reads the other buffer any more
        if (kv0 + KT < hi) {
#pragma unroll
          for (int kg = 0; kg < KT / 16; ++kg) ask(next[kg], kv0 + KT + 16 * kg);
          fetch(kv0 + KT, buf ^ 1);
        }
#pragma unroll
        for (int kg = 0; kg < KT / 16; ++kg) {
          const int c0 = kv0 + 16 * kg;
          if (!block_live<true>(p, r0, s.n_q, c0, hi)) continue;
          float bias[4] = {0.f, 0.f, 0.f, 0.f};
          int bucket[4] = {0, 0, 0, 0};
          const uint32_t keep = pairs(ta, tlp, now[kg].raw, c0, g, bias, bucket);
          if (__builtin_amdgcn_ballot_w64(keep != 0u) == 0) continue;
          floatx4 x;
#pragma unroll
          for (int r = 0; r < 4; ++r) x[r] = now[kg].x[r] * p.inv_n;
          dot_cols<D>(o, sm + buf * TILE_F, 16 * kg, m, g, x);
          bias_grads<TAB, DEN>(p, tlp, diag + (c0 - lo) + 4 * g + (TILE - 1) - (WROWS * w + m), dsm, x, bucket, want_pos, want_ts, b, r0, c0, m, g, w, lane);
        }
      }
      bias_grads_out<TAB>(p, ta, tlp, diag, n_diag, want_pos, want_ts, h, lo, q0, tid);
    }
  }
  if (qi < s.rows)
    store_row<float, D>((float*)p.dq + s.bq + (int64_t)qi * p.q_st, o, qi < s.n_q ? p.alpha : 0.f, g);
}

template <typename T, int D, bool TAB, bool DEN>
__global__ __launch_bounds__(256, D >= 128 ? 2 : 3) void hstu_f32_dkv(const Params p, const TabArg<TAB> ta) {
  using S = Shape<D>;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  __shared__ typename std::conditional<TAB, TabLds, Nothing>::type tl;
  const int h = blockIdx.x, b = blockIdx.y, kt = blockIdx.z;
  const Seq s = seq_info(p, b, h);
  const int k0 = kt * TILE;
  const int rows = p.jagged ? s.rows : p.Lkv;
  if (k0 >= rows) return;
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = k0 + WROWS * w, kj = r0 + m;
  floatx4 ok[S::NS], ov[S::NS];
#pragma unroll
  for (int x = 0; x < S::NS; ++x) { ok[x] = floatx4{0.f, 0.f, 0.f, 0.f}; ov[x] = floatx4{0.f, 0.f, 0.f, 0.f}; }
  if (k0 < s.n_kv) {
    int lo, hi;
    query_range<DEN>(p, s, b, k0, tid, lo, hi);
    if (lo < hi) {
      const Tiles<T, D> t = {(const T*)p.q + s.bq, (const T*)p.dout + s.bo, (int)(p.q_st * sizeof(T)), (int)(p.o_st * sizeof(T)), s.n_q, w, lane, sm};
      t.fetch(lo, 0);
      float4 kf[S::NS], vf[S::NS];
      {
        const int kc = kj < s.n_kv ? kj : s.n_kv - 1;
        const T* krow = (const T*)p.k + s.bk + (int64_t)kc * p.k_st + 4 * g;
        const T* vrow = (const T*)p.v + s.bv + (int64_t)kc * p.v_st + 4 * g;
#pragma unroll
        for (int x = 0; x < S::NS; ++x) { kf[x] = load4(krow + 16 * x); vf[x] = load4(vrow + 16 * x); }
      }
      if constexpr (TAB) {
        if (p.ts_tab) tab_setup(p, ta, tl, h, tid);
      }
      Pairs<TAB, DEN, false> pairs(p, s, b, h, kj);
      float* const dsg = sizeof(T) == 4 && p.ds ? ds_blocks(p, b, h, s) + 16 * m + 4 * g : nullptr;
      const TabLds* tlp = nullptr;
      if constexpr (TAB) tlp = &tl;
      typename decltype(pairs)::Raw raw[S::KG], next[S::KG];
#pragma unroll
      for (int kg = 0; kg < S::KG; ++kg) pairs.load(next[kg], lo + 16 * kg, g);
      int buf = 0;
      for (int i0 = lo; i0 < hi; i0 += S::KT, buf ^= 1) {
        dma_wait();
#pragma unroll
        for (int kg = 0; kg < S::KG; ++kg) { next[kg].arrived(); raw[kg] = next[kg]; }
        __syncthreads();              // the step's tiles are there, and nobody reads the other buffer any more
        if (i0 + S::KT < hi) {
#pragma unroll
          for (int kg = 0; kg < S::KG; ++kg) pairs.load(next[kg], i0 + S::KT + 16 * kg, g);
          t.fetch(i0 + S::KT, buf ^ 1);
        }
#pragma unroll
        for (int kg = 0; kg < S::KG; ++kg) {
          const int c0 = i0 + 16 * kg;
          if (!block_live<false>(p, r0, s.n_kv, c0, hi)) continue;
          float bias[4] = {0.f, 0.f, 0.f, 0.f};
          int bucket[4];
          const uint32_t keep = pairs(ta, tlp, raw[kg], c0, g, bias, bucket);
          if (__builtin_amdgcn_ballot_w64(keep != 0u) == 0) continue;
          floatx4 x, dp, pr;
          dot_rows2<D>(x, dp, t.tile(buf, 0), t.tile(buf, 1), 16 * kg + m, g, kf, vf);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float u = p.alpha * x[r];
            if constexpr (TAB || DEN) u += bias[r];
            const float sg = sigmoid(u);
            pr[r] = kept(u * sg, keep, r);
            x[r] = kept(dp[r] * sg * (1.0f + u * (1.0f - sg)), keep, r);
          }
          if (sizeof(T) == 4 && D >= 32 && dsg) __builtin_nontemporal_store(x, (floatx4*)(dsg + ds_block_at(p, c0 >> 4, r0 >> 4)));
          dot_cols<D>(ov, t.tile(buf, 1), 16 * kg, m, g, pr);
          dot_cols<D>(ok, t.tile(buf, 0), 16 * kg, m, g, x);
        }
      }
    }
  }
  if (kj < rows) {
    const bool live = kj < s.n_kv;
    store_row<T, D>((T*)p.dk + s.bk + (int64_t)kj * p.k_st, ok, live ? p.alpha * p.inv_n : 0.f, g);
    store_row<T, D>((T*)p.dv + s.bv + (int64_t)kj * p.v_st, ov, live ? p.inv_n : 0.f, g);
  }
}

// ---------------------------------------------------------------------------
// Dispatch
// ---------------------------------------------------------------------------

bool rows_whole(const void* base, int64_t row, int64_t head, int64_t batch, int bytes) {
  return ((uintptr_t)base & (uintptr_t)(4 * bytes - 1)) == 0 && ((row | head | batch) & 3) == 0;
}

template <bool TAB>
TabArg<TAB> tab_arg(const Params& p) {
  TabArg<TAB> ta;
  memset(&ta, 0, sizeof(ta));
  if constexpr (TAB) {
    if (p.ts_tab) {
      const int32_t* thr;
      const int reach = bucket_thresholds(p.ts_bucket_size, &thr);
      memcpy(ta.thr, thr, sizeof(ta.thr));
      ta.per_log2 = LN2 / p.ts_bucket_size;
      ta.top = p.ts_nb < reach ? p.ts_nb : reach;
    }
  }
  return ta;
}

int launched(const char* what) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? HSTU_OK : fail(HSTU_ERR_LAUNCH, "%s launch: %s", what, hipGetErrorString(e));
}

template <typename T, int D, bool TAB, bool DEN>
int fwd_inst(const Params& p, hipStream_t st) {
  const dim3 grid(p.H, p.B, (p.L + TILE - 1) / TILE);
  hipLaunchKernelGGL((hstu_f32_fwd<T, D, TAB, DEN>), grid, dim3(256), sizeof(float) * Shape<D>::LDS_F, st, p, tab_arg<TAB>(p));
  return launched("fp32 forward kernel");
}
template <typename T, int D, bool TAB, bool DEN>
int bwd_inst(const Params& p, hipStream_t st) {
  const size_t smem = sizeof(float) * Shape<D>::LDS_F;
  const bool want_pos = TAB && p.dpos && p.pos_tab;
  const dim3 grid_q(p.H, p.B, (p.L + TILE - 1) / TILE), grid_k(p.H, p.B, (p.Lkv + TILE - 1) / TILE);
  const TabArg<TAB> ta = tab_arg<TAB>(p);
  if constexpr (sizeof(T) == 4 && D >= 32) {
    if (p.ds) {
      hipLaunchKernelGGL((hstu_f32_dkv<T, D, TAB, DEN>), grid_k, dim3(256), smem, st, p, ta);
      if (int rc = launched("fp32 backward dk/dv kernel")) return rc;
      const size_t smem_q = sizeof(float) * (2 * 32 * D + (want_pos ? ((p.Lkv + 15) & ~15) + TILE + 32 : 0));
      hipLaunchKernelGGL((hstu_f32_dq_ds<D, TAB, DEN>), grid_q, dim3(256), smem_q, st, p, ta);
      return launched("fp32 backward dq kernel");
    }
  }
  hipLaunchKernelGGL((hstu_f32_dq<T, D, TAB, DEN>), grid_q, dim3(256), smem + (want_pos ? sizeof(float) * (((p.Lkv + 15) & ~15) + TILE + 32) : 0), st, p, ta);
  if (int rc = launched("fp32 backward dq kernel")) return rc;
  hipLaunchKernelGGL((hstu_f32_dkv<T, D, TAB, DEN>), grid_k, dim3(256), smem, st, p, ta);
  return launched("fp32 backward dk/dv kernel");
}
template <typename T, int D>
int launch_d(const Params& p, bool bwd, hipStream_t st) {
  const bool tab = p.pos_tab || p.ts_tab, den = p.mask || p.dense_bias;
  if (tab) return bwd ? bwd_inst<T, D, true, false>(p, st) : fwd_inst<T, D, true, false>(p, st);
  if (den) return bwd ? bwd_inst<T, D, false, true>(p, st) : fwd_inst<T, D, false, true>(p, st);
  return bwd ? bwd_inst<T, D, false, false>(p, st) : fwd_inst<T, D, false, false>(p, st);
}
int launch(const Params& p, bool bf16, bool bwd, hipStream_t st) {
  if (bf16) return launch_d<bf16_t, 16>(p, bwd, st);
  switch (p.d_qk) {
    case 128: return launch_d<float, 128>(p, bwd, st);
    case 64: return launch_d<float, 64>(p, bwd, st);
    case 32: return launch_d<float, 32>(p, bwd, st);
    default: return launch_d<float, 16>(p, bwd, st);
  }
}

}  // namespace

// Not theirs, and left to the general kernels: other head dims; rows that cannot be fetched four elements at a time; a table
// and a dense operand in one call; tables of lengths whose position sums exceed LDS; bucket sizes with more than 256 buckets.
bool hstu::f32_takes(const Params& p, bool bf16, bool backward) {
  const int bytes = bf16 ? 2 : 4;
  if (p.d_qk != p.d_v || !(p.d_qk == 16 || (!bf16 && (p.d_qk == 32 || p.d_qk == 64 || p.d_qk == 128)))) return false;
  if (!rows_whole(p.q, p.q_st, p.q_sh, p.q_sb, bytes) || !rows_whole(p.k, p.k_st, p.k_sh, p.k_sb, bytes) ||
      !rows_whole(p.v, p.v_st, p.v_sh, p.v_sb, bytes)) return false;
  if (backward ? !(rows_whole(p.dout, p.o_st, p.o_sh, p.o_sb, bytes) && rows_whole(p.dq, 0, 0, 0, bytes) && rows_whole(p.dk, 0, 0, 0, bytes) &&
                   rows_whole(p.dv, 0, 0, 0, bytes))
               : !rows_whole(p.out, p.o_st, p.o_sh, p.o_sb, bytes)) return false;
  for (int64_t st : {p.q_st, p.k_st, p.v_st, p.o_st})
    if (st < 0 || st * bytes >= (1LL << 31)) return false;
  const bool tab = p.pos_tab || p.ts_tab, den = p.mask || p.dense_bias;
  if (tab && (den || p.L > TAB_MAX_L)) return false;
  if (p.ts_tab) {
    const int32_t* thr;
    if (bucket_thresholds(p.ts_bucket_size, &thr) + 2 >= LAW_THR_LEN) return false;
  }
  if (p.mask && p.Lkv < 4) return false;
  return p.B <= 65535 && (p.L + TILE - 1) / TILE <= 65535 && (p.Lkv + TILE - 1) / TILE <= 65535;
}
// Bytes for the blocks of dS of a backward call (see ds_blocks), 0 where both kernels form them.  Kept, two of the dQ kernel's three products and
// its activation go, for 4 bytes a pair and head written and read.  us for a backward call, formed twice -> kept:
//   d = 128: 128 x 512 1490 -> 1191 (segment ids), 2261 -> 1731; 32 x up to 1024 with the position table 1189 -> 868; 32 x 128, four heads
//            51 -> 41
//   d = 64:  128 x 512 747 -> 609 (segment ids); 64 x 512 with the table 717 -> 603; 8 x 2048, both tables 1677 -> 1394; 16 x 256 52 -> 42
//   d = 32:  128 x 512 654 -> 572; 8 x 2048, both tables 1173 -> 999; 16 x 256, four heads 36 -> 32; 32 x 128 and 4 x 64 27 -> 28
//   a window's band, eight heads: 16 x 2048, window 256: d = 128 1163 -> 881, d = 64 590 -> 454, d = 32 317 -> 262; 8 x 256, four heads, window
//            32: d = 128 38 -> 31, d = 64 27 -> 27
// Those of 27 us are as long as their launches and the host's work: the line below leaves such calls (and head dims of 16) alone.
size_t hstu::f32_ds_bytes(const Params& p, int64_t total_tokens, int64_t* per_head, DsRows* in_head) {
  const int64_t nq = (p.L + 15) / 16, nk = (p.Lkv + 15) / 16, rows = p.jagged ? (total_tokens >> 4) + p.B : (int64_t)p.B * nq;
  const DsRows slots = ds_row_slots(nq, nk, p.causal && p.L == p.Lkv, p.causal != 0, p.window, 16);
  const double bytes = (double)rows * slots.per_row * (4.0 * DS_BLOCK) * p.H;
  if (p.d_qk < 32 || bytes * p.d_qk < 2e8 || bytes > (double)DS_MAX_BYTES) return 0;
  if (per_head) { *per_head = rows * slots.per_row * (4 * DS_BLOCK); *in_head = slots; }
  return (size_t)(rows * slots.per_row * (4 * DS_BLOCK)) * p.H;
}
int hstu::f32_launch_fwd(const Params& p, bool bf16, hipStream_t st) { return launch(p, bf16, false, st); }
int hstu::f32_launch_bwd(const Params& p, bool bf16, hipStream_t st) { return launch(p, bf16, true, st); }
