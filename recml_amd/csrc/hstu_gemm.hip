// The matrix products of an HSTU block on the matrix cores of gfx950, in bf16 with fp32 accumulation.
//
//   HSTU_GEMM_NN   out[m, n] = act(sum_k x[m, k] w[k, n] + bias[n] + c[m, n])     a projection
//   HSTU_GEMM_NT   out[m, k] = sum_n x[m, n] w[k, n]                              the gradient of its input
//   HSTU_GEMM_TN   out[k, n] = sum_m x[m, k] y[m, n]                              the gradient of its weight
//
// The weight (NN, NT) and the weight's gradient (TN) may come as several matrices side by side along n ("slabs": the
// U, Q, K and V kernels of a block), so nobody concatenates them.  See hstu_gemm_kernel for the layout of the work.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "hstu_block.h"
#include "hstu_block_common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v* lds_short4_ptr;

constexpr int GEMM_BK = 32;          // contraction depth of a stage

struct GemmParams {
  const bf16_t* q;                   // the operand of the output's rows
  const bf16_t* p[HSTU_GEMM_MAX_SLABS];   // the operand of its columns, as slabs
  bf16_t* out[HSTU_GEMM_MAX_SLABS];
  float* partial;                    // split contraction: [split][rows][cols] sums instead of `out`
  bf16_t* pre;                       // the value before the activation is stored here as well (or null)
  const bf16_t* bias;
  const bf16_t* c;
  const bf16_t *gamma, *beta;             // (hstu_gemm_rows_kernel: the rows' layer norm, or null)
  float eps;
  int64_t q_stride, p_stride, out_stride, c_stride;
  int32_t rows, cols, depth;         // of the product: output rows and columns, contraction
  int32_t slab, out_slab;            // width of a slab of `p` (along the weight's n) and of `out` (along its columns)
  int32_t splits, depth_per_split;
  int32_t row_tiles, col_tiles;
  int32_t activation;
};

// 256 bytes of zeros: what lanes whose element lies outside an operand load.
__device__ __attribute__((aligned(256))) unsigned char gemm_zeros[256];

__device__ __forceinline__ void lds_dma16(const void* src, uint32_t lds_addr_wave_uniform) {
  const uint32_t base = __builtin_amdgcn_readfirstlane(lds_addr_wave_uniform);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(base), "v"(src) : "memory", "m0");
}

// The same with a scalar base and a 32-bit lane offset.
__device__ __forceinline__ void lds_dma16(const char* base_uniform, uint32_t off, uint32_t lds_addr_wave_uniform) {
  const uint32_t to = __builtin_amdgcn_readfirstlane(lds_addr_wave_uniform);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(to), "v"(off), "s"(base_uniform) : "memory", "m0");
}
__device__ __forceinline__ const char* scalar_ptr(const void* p) {
  const uint64_t v = (uint64_t)(uintptr_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const char*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

#define HSTU_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt((((n) & 15) | ((((n) >> 4) & 3) << 14)) | 0x0F70)

// 16 bytes of the output.  PAST: not kept in this XCD's L2, where the operands are (the reader is a later launch, on any XCD).  store_past
// says for which outputs.
template <bool PAST>
__device__ __forceinline__ void store_out(bf16_t* to, const uint4& v) {
  typedef uint32_t words __attribute__((ext_vector_type(4)));
  const words x = {v.x, v.y, v.z, v.w};
  if constexpr (PAST) __builtin_nontemporal_store(x, (words*)to);
  else *(words*)to = x;
}

// Whether an output of these sizes is stored past the L2s: where it is larger than all of them together (32 MB), so that it would drive the
// operands out and its reader would not find it there, and its rows are whole sectors of 64 bytes.  us with / without:
//   74 k x 512 -> 2048 190 / 217, with the pre-activation 226 / 282; 78 k x 512 -> 512 57 / 59; 78 k x 64 -> 256 (40 MB) 12.3 / 14.7
//   1600 x 64 -> 20000 (64 MB) 22.7 / 25.7
//   rows of parts of sectors, which leave as parts of lines: 8000 x 64 -> 5000 39 / 27, 16384 x 1024 -> 1000 44 / 37
//   below 32 MB the product gains what its reader loses (18 k x 64 -> 128 with a pass over the result 9.7 / 9.7, 6.4 k x 512 -> 2048 30.9 / 31.2;
//   an attention behind 18 k rows of 128 28.7 / 27.3)
bool store_past(int64_t rows, int64_t cols, int64_t stride) { return rows * cols > 16 << 20 && stride % 32 == 0; }

// One workgroup: a tile of 64 MB output rows x 32 NB WN output columns, 2 x WN waves of 32 MB x 32 NB.  The contraction runs in
// stages of 32 through a three-stage LDS ring filled by direct global -> LDS loads (two stages in flight, one barrier
// per stage).  The product is formed transposed (columns as the matrix instruction's rows): a lane then holds four
// consecutive columns of one output row.
//   An operand stored along the contraction (Q_T / P_T false) lies in LDS as rows of 64 bytes, 16-byte chunk c of row r at
// c ^ (r / 4 % 4): a fragment is one ds_read_b128 per lane, 16 rows reach all 64 banks.  One stored across it (x and dz in
// the weight's gradient, the weight itself in the forward) lies as 32 rows of 128 columns, chunk c at c ^ 4 (r % 4), and is
// transposed on the way out by ds_read_b64_tr_b16, two per fragment.
//   Why 128 x 64 per wave (MB 4, NB 2): with 64 x 64 the four SIMDs' fragments take all of the LDS bandwidth (128 bytes a clock) at
// full matrix rate, with 128 x 64 three quarters of it, and the direct loads' writes come on top: 72 KB per 512 clocks in a tile of
// 256 x 128, 131 KB per 1024 in one of 256 x 256 (WN 4), whose main loop is the faster one (1290 against 1100 TFLOP/s over long
// contractions); 256 x 128 leaves two workgroups per CU, so that one's stores run under the other's products.  Without its epilogue
// 74 k x 512 -> 2048 takes 139 us, with it 194: the stores burst at a tile's end.
//   UNIFORM: a tile's columns of P (a stage's, where P lies along the contraction) are in one slab.  A load is then a scalar base
// that moves on with the stage and a lane offset that never changes; rows and columns past an operand's end repeat its last
// (what they give is not stored), and only the stage that crosses the contraction's end tests its elements.  Per-lane
// pointers, counters and slab hops were three of the ten vector instructions behind every matrix instruction.
//   OUT: what the epilogue does, known to the compiler where it is one of the products of a block: a branch between its steps keeps
// it from ordering them across pieces (74 k x 512 -> 2048 with the activation 235 us, 194 without).
enum { OUT_PLAIN, OUT_SILU, OUT_PRE_SILU, OUT_ADD, OUT_PARTIAL, OUT_ANY };
template <int MB, int NB, int WN, bool Q_T, bool P_T, int STAGES, bool UNIFORM, int OUT, bool PAST>
__global__ __launch_bounds__(128 * WN, 2) void hstu_gemm_kernel(const GemmParams g) {
  constexpr int TM = 64 * MB, TN = 32 * NB * WN, WAVES = 2 * WN;
  constexpr int Q_BYTES = TM * GEMM_BK * 2, P_BYTES = TN * GEMM_BK * 2, STAGE = Q_BYTES + P_BYTES;
  constexpr int LQ = Q_BYTES / (1024 * WAVES), LP = P_BYTES / (1024 * WAVES);      // direct loads of 1 KB per wave
  static_assert(LQ >= 1 && LP >= 1, "a stage is at least one load per wave and operand");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const uint32_t smem_lds = __builtin_amdgcn_groupstaticsize();
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;

  // Workgroups go to the eight XCDs in turn: the column tiles of a row tile (which share the row operand) follow each
  // other on one XCD; with a split contraction all tiles of a split do.
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
  int rt, ct, split = 0;
  if (g.splits > 1) {
    // (fewer splits than XCDs, 2 or 4: each has 4 or 2 of them, which take its tiles in turn)
    const int per = g.row_tiles * g.col_tiles;
    int t;
    if (g.splits < 8) {
      split = xcd & (g.splits - 1);
      t = j * (8 / g.splits) + xcd / g.splits;
      if (t >= per) return;
    } else {
      split = (j / per) * 8 + xcd;
      t = j % per;
      if (split >= g.splits) return;
    }
    rt = t / g.col_tiles;
    ct = t - rt * g.col_tiles;
  } else {
    rt = (j / g.col_tiles) * 8 + xcd;
    ct = j % g.col_tiles;
    if (rt >= g.row_tiles) return;
  }
  const int m0 = rt * TM, n0 = ct * TN;
  const int k_begin = split * g.depth_per_split;
  const int k_end = k_begin + g.depth_per_split < g.depth ? k_begin + g.depth_per_split : g.depth;
  const int nt = (k_end - k_begin + GEMM_BK - 1) / GEMM_BK;

  // ---- what each lane loads: piece i of an operand is 1 KB of LDS, lane l of it 16 bytes at 16 l.
  //   along:  row = 16 piece + l / 4, physical chunk l % 4           (advance: 32 elements per stage)
  //   across: panel of 128 columns, row = 4 (piece % 8) + l / 16, physical chunk l % 16    (advance: 32 rows per stage)
  // A source past the operand's end is the page of zeros.
  // Small tiles (64 columns) across the contraction: rows of 64 columns, 8 rows per piece, chunk c at c ^ 4 (r / 2 % 2).
  struct Src { int outer, k; };      // index along the output's axis, and along the contraction
  auto src_of = [&](bool across, int tile, int piece) {
    Src s;
    if (!across) {
      const int row = 16 * piece + (lane >> 2);
      s.outer = row;
      s.k = 8 * ((lane & 3) ^ ((row >> 2) & 3));
    } else if (tile >= 128) {
      const int panel = piece >> 3, row = 4 * (piece & 7) + (lane >> 4);
      s.outer = 128 * panel + 8 * ((lane & 15) ^ (4 * (row & 3)));
      s.k = row;
    } else {
      const int row = 8 * piece + (lane >> 3);
      s.outer = 8 * ((lane & 7) ^ (4 * ((row >> 1) & 1)));
      s.k = row;
    }
    return s;
  };
  const char* qp[LQ];
  const char* pp[LP];
  int qk[LQ], pk[LP];                // contraction index of the lane's next load; past k_end: zeros
  int ps[LP], pc[LP];                // P along the contraction in slabs: slab and column within it
  int po[LP];
#pragma unroll
  for (int i = 0; i < LQ; ++i) {
    const Src s = src_of(Q_T, TM, w * LQ + i);
    const int m = m0 + s.outer;
    qk[i] = m < g.rows ? k_begin + s.k : 0x3fffffff;
    qp[i] = (const char*)(Q_T ? g.q + (int64_t)(k_begin + s.k) * g.q_stride + m : g.q + (int64_t)m * g.q_stride + k_begin + s.k);
  }
#pragma unroll
  for (int i = 0; i < LP; ++i) {
    const Src s = src_of(P_T, TN, w * LP + i);
    const int n = n0 + s.outer;
    pk[i] = n < g.cols ? k_begin + s.k : 0x3fffffff;
    if (P_T) {
      // across the contraction: the column decides the slab, once (TN: y is one matrix, its slab the whole width)
      const int sl = n < g.cols ? n / g.slab : 0;
      pp[i] = (const char*)(g.p[sl] + (int64_t)(k_begin + s.k) * g.p_stride + (n - sl * g.slab));
      ps[i] = pc[i] = po[i] = 0;
    } else {
      ps[i] = (k_begin + s.k) / g.slab;
      pc[i] = k_begin + s.k - ps[i] * g.slab;
      po[i] = n;
      const int sl = ps[i] < HSTU_GEMM_MAX_SLABS ? ps[i] : 0;
      pp[i] = (const char*)((sl == 0 ? g.p[0] : sl == 1 ? g.p[1] : sl == 2 ? g.p[2] : g.p[3]) + (int64_t)n * g.p_stride + pc[i]);
    }
  }
  // (UNIFORM: lane offsets; the scalar bases follow from the stage)
  uint32_t qo[LQ], uo[LP];
  const char *q_base = nullptr, *p_base = nullptr;
  int u_k = k_begin, u_slab = 0, u_col = 0;      // contraction index of the next stage to load; P along it: its slab and column there
  if constexpr (UNIFORM) {
#pragma unroll
    for (int i = 0; i < LQ; ++i) {
      Src s = src_of(Q_T, TM, w * LQ + i);
      const int most = g.rows - (Q_T ? 8 : 1) - m0;
      s.outer = s.outer < most ? s.outer : most;
      qo[i] = Q_T ? (uint32_t)(s.k * (int)g.q_stride + s.outer) * 2u : (uint32_t)(s.outer * (int)g.q_stride + s.k) * 2u;
      qk[i] = s.k;
    }
#pragma unroll
    for (int i = 0; i < LP; ++i) {
      Src s = src_of(P_T, TN, w * LP + i);
      const int most = g.cols - (P_T ? 8 : 1) - n0;
      s.outer = s.outer < most ? s.outer : most;
      uo[i] = P_T ? (uint32_t)(s.k * (int)g.p_stride + s.outer) * 2u : (uint32_t)(s.outer * (int)g.p_stride + s.k) * 2u;
      pk[i] = s.k;
    }
    q_base = scalar_ptr(Q_T ? g.q + (int64_t)k_begin * g.q_stride + m0 : g.q + (int64_t)m0 * g.q_stride + k_begin);
    if (P_T) {
      const int sl = n0 / g.slab;
      p_base = scalar_ptr(g.p[sl] + (int64_t)k_begin * g.p_stride + (n0 - sl * g.slab));
    } else {
      u_slab = k_begin / g.slab;
      u_col = k_begin - u_slab * g.slab;
      p_base = scalar_ptr(g.p[u_slab] + (int64_t)n0 * g.p_stride + u_col);
    }
  }
  const int64_t q_step = Q_T ? (int64_t)GEMM_BK * g.q_stride * 2 : GEMM_BK * 2;
  const int64_t p_step = (int64_t)GEMM_BK * g.p_stride * 2;
  constexpr int NLOAD = LQ + LP;     // of a stage, per wave
  auto issue_one = [&](int st, int i) {
    const uint32_t base = smem_lds + (uint32_t)st * STAGE;
    if constexpr (UNIFORM) {
      const bool whole = u_k + GEMM_BK <= k_end;
      const uint32_t to = i < LQ ? base + 1024u * (w * LQ + i) : base + Q_BYTES + 1024u * (w * LP + i - LQ);
      const char* from = i < LQ ? q_base : p_base;
      const uint32_t off = i < LQ ? qo[i < LQ ? i : 0] : uo[i < LQ ? 0 : i - LQ];
      if (whole) {
        lds_dma16(from, off, to);
      } else {
        const int k = u_k + (i < LQ ? qk[i < LQ ? i : 0] : pk[i < LQ ? 0 : i - LQ]);
        lds_dma16(k < k_end ? (const void*)(from + off) : (const void*)(gemm_zeros + 16 * (lane & 15)), to);
      }
      if (i == NLOAD - 1) {       // on to the next stage (past the end the bases stay: everything there is zeros)
        u_k += GEMM_BK;
        if (u_k < k_end) {
          q_base += q_step;
          if (P_T) {
            p_base += p_step;
          } else {
            u_col += GEMM_BK;
            p_base += GEMM_BK * 2;
            if (u_col >= g.slab) {
              u_col = 0;
              ++u_slab;
              p_base = scalar_ptr(g.p[u_slab] + (int64_t)n0 * g.p_stride);
            }
          }
        }
      }
      return;
    }
    if (i < LQ) {
      const void* src = qk[i] < k_end ? (const void*)qp[i] : (const void*)(gemm_zeros + 16 * (lane & 15));
      lds_dma16(src, base + 1024u * (w * LQ + i));
      qp[i] += q_step;
      qk[i] += GEMM_BK;
      return;
    }
    i -= LQ;
    const void* src = pk[i] < k_end ? (const void*)pp[i] : (const void*)(gemm_zeros + 16 * (lane & 15));
    lds_dma16(src, base + Q_BYTES + 1024u * (w * LP + i));
    pk[i] += GEMM_BK;
    if (P_T) {
      pp[i] += p_step;
    } else {
      // along the contraction, and on to the next slab where this one ends (selects: a branch here would cut the products
      // around it into separate schedules)
      pc[i] += GEMM_BK;
      const bool over = pc[i] >= g.slab;
      pc[i] -= over ? g.slab : 0;
      const int64_t hop = ps[i] == 0 ? g.p[1] - g.p[0] : ps[i] == 1 ? g.p[2] - g.p[1] : g.p[3] - g.p[2];
      pp[i] += GEMM_BK * 2 + (over ? (hop - g.slab) * 2 : 0);
      ps[i] += over ? 1 : 0;
    }
  };

  // ---- fragments: lane (index l32 of a block of 32, half hh) holds contraction elements 16 s + 8 hh .. + 7
  const int wm = w & 1, wn = w >> 1;
  const int gi = lane & 15;
  auto frag = [&](bool across, int tile, const unsigned char* base, int block, int s) -> bf16x8 {
    if (!across) {
      const int r = 32 * block + l32;
      return *(const bf16x8*)(base + r * 64 + (((2 * s + hh) ^ ((r >> 2) & 3)) * 16));
    }
    const int row = 16 * s + 8 * hh + (gi >> 2);
    const int c2 = 2 * ((lane >> 4) & 1) + ((gi & 3) >> 1);
    const unsigned char* at;
    int pitch;
    if (tile >= 128) {
      const int panel = block >> 2, ob = block & 3;
      pitch = 256;
      at = base + panel * (GEMM_BK * 256) + row * 256 + (4 * (ob ^ (gi >> 2)) + c2) * 16 + 8 * (gi & 1);
    } else {
      pitch = 128;
      at = base + row * 128 + ((4 * ((block & 1) ^ ((row >> 1) & 1)) + c2)) * 16 + 8 * (gi & 1);
    }
    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(at));
    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(at + 4 * pitch));
    struct { short4v a, b; } both = {lo, hi};
    return __builtin_bit_cast(bf16x8, both);
  };

  floatx16 acc[NB][MB];
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;

  static_assert((STAGES - 1) * NLOAD <= 63 && STAGES >= 2 && STAGES <= 4, "vmcnt range");
  struct Frags { bf16x8 p[NB], q[MB]; };
  auto load = [&](int st, int s, Frags& f) {
    const unsigned char* qb = smem + st * STAGE;
    const unsigned char* pb = qb + Q_BYTES;
#pragma unroll
    for (int a = 0; a < NB; ++a) f.p[a] = frag(P_T, TN, pb, wn * NB + a, s);
#pragma unroll
    for (int b = 0; b < MB; ++b) f.q[b] = frag(Q_T, TM, qb, wm * MB + b, s);
  };
  // One sub-step's products; with `refill` the loads of the stage that takes place `st` go out between them: issued
  // back to back they would hold the wave up (the CU's memory front end takes one every 16 cycles from all its waves).
  auto products = [&](const Frags& f, auto refill_, int st) {
    constexpr bool refill = decltype(refill_)::value;
    int next = 0;
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int a = 0; a < NB; ++a) {
        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.p[a], f.q[b], acc[a][b], 0, 0, 0);
        if constexpr (refill) {
          const int due = ((b * NB + a + 1) * NLOAD) / (MB * NB);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < NLOAD; ++i)
            if (i >= next && i < due) issue_one(st, i);
          __builtin_amdgcn_sched_barrier(0);
          next = due;
        }
      }
  };
  // Stages past the contraction's end are loaded too (zeros), so that every wait counts the same number of younger loads.
#pragma unroll
  for (int t = 0; t < STAGES; ++t)
#pragma unroll
    for (int i = 0; i < NLOAD; ++i) issue_one(t, i);
  // A stage's two sub-steps of 16: the fragments of each are asked for ahead of the products of the one before it, so that
  // the matrix pipe has work while they come.  The order is fixed by scheduling barriers.
  Frags fa, fb;
  HSTU_WAIT_VMCNT((STAGES - 1) * NLOAD);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  load(0, 0, fa);
  int st = 0;
  for (int t = 0; t < nt; ++t) {
    load(st, 1, fb);
    __builtin_amdgcn_sched_barrier(0);
    products(fa, std::false_type{}, 0);
    __builtin_amdgcn_sched_barrier(0);
    // (fb is here: the stage's last read is done, and behind the barrier everyone's is: its place can be refilled)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    HSTU_WAIT_VMCNT((STAGES - 2) * NLOAD);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int next = st + 1 >= STAGES ? 0 : st + 1;
    load(next, 0, fa);
    __builtin_amdgcn_sched_barrier(0);
    products(fb, std::true_type{}, st);
    __builtin_amdgcn_sched_barrier(0);
    st = next;
  }
  HSTU_WAIT_VMCNT(0);
  __syncthreads();

  // ---- out: blocks of 32 rows x 32 NB columns through the wave's own LDS (fp32, rows 16 bytes apart from a multiple of 256:
  // conflict-free both ways), then whole row pieces of 8 columns per lane
  constexpr int W = 32 * NB, PITCH = W * 4 + 16;
  unsigned char* stage = smem + w * (32 * PITCH);
  constexpr int LPR = W / 8, RPI = 64 / LPR;        // lanes per row, rows per instruction
  const int rr = lane / LPR, cc = lane - rr * LPR;
  const int n = n0 + wn * W + 8 * cc;
  float bias[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) bias[i] = 0.f;
  if (g.bias && n < g.cols) unpack8(*(const uint4*)(g.bias + n), bias);
  const int osl = (g.partial || n >= g.cols) ? 0 : n / g.out_slab;
#pragma unroll
  for (int b = 0; b < MB; ++b) {
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const float4 v = {acc[a][b][4 * q4], acc[a][b][4 * q4 + 1], acc[a][b][4 * q4 + 2], acc[a][b][4 * q4 + 3]};
        *(float4*)(stage + l32 * PITCH + (32 * a + 8 * q4 + 4 * hh) * 4) = v;
      }
    __builtin_amdgcn_wave_barrier();
    // (the steps below over all pieces of the block at a time: a piece by itself is a chain of dependent transcendentals with
    // nothing beside it, 240 us where this takes 204 at 74 k x 512 -> 2048)
    constexpr int PIECES = 32 / RPI;
    float x[PIECES][8];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const unsigned char* at = stage + (RPI * i + rr) * PITCH + 32 * cc;
      const float4 v0 = *(const float4*)at, v1 = *(const float4*)(at + 16);
      x[i][0] = v0.x; x[i][1] = v0.y; x[i][2] = v0.z; x[i][3] = v0.w;
      x[i][4] = v1.x; x[i][5] = v1.y; x[i][6] = v1.z; x[i][7] = v1.w;
    }
    const int mb = m0 + wm * 32 * MB + 32 * b + rr;      // the lane's row of piece 0
    auto inside = [&](int i) { return mb + RPI * i < g.rows && n < g.cols; };
    if constexpr (OUT == OUT_PARTIAL) {
#pragma unroll
      for (int i = 0; i < PIECES; ++i)
        if (inside(i)) {
          float* o = g.partial + ((int64_t)split * g.rows + mb + RPI * i) * g.cols + n;
          *(float4*)o = float4{x[i][0], x[i][1], x[i][2], x[i][3]};
          *(float4*)(o + 4) = float4{x[i][4], x[i][5], x[i][6], x[i][7]};
        }
    } else {
      if (OUT == OUT_ADD || (OUT == OUT_ANY && g.c)) {
        uint4 cr[PIECES];
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
          cr[i] = uint4{0u, 0u, 0u, 0u};
          if (inside(i)) cr[i] = *(const uint4*)(g.c + (int64_t)(mb + RPI * i) * g.c_stride + n);
        }
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
          float cv[8];
          unpack8(cr[i], cv);
#pragma unroll
          for (int e = 0; e < 8; ++e) x[i][e] += cv[e];
        }
      }
      if (!Q_T && P_T) {        // (zeros without one)
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) x[i][e] += bias[e];
      }
      if (OUT == OUT_PRE_SILU || (OUT == OUT_ANY && g.pre)) {
        // (the activation of the stored value, which is what its gradient is taken at)
#pragma unroll
        for (int i = 0; i < PIECES; ++i) {
          const uint4 z = pack8(x[i]);
          if (inside(i)) store_out<PAST>(g.pre + (int64_t)(mb + RPI * i) * g.out_stride + n, z);
          unpack8(z, x[i]);
        }
      }
      if (OUT == OUT_SILU || OUT == OUT_PRE_SILU || (OUT == OUT_ANY && g.activation)) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) x[i][e] = silu(x[i][e]);
      }
      bf16_t* o = (osl == 0 ? g.out[0] : osl == 1 ? g.out[1] : osl == 2 ? g.out[2] : g.out[3]) + (int64_t)mb * g.out_stride + (n - osl * g.out_slab);
#pragma unroll
      for (int i = 0; i < PIECES; ++i)
        if (inside(i)) store_out<PAST>(o + (int64_t)(RPI * i) * g.out_stride, pack8(x[i]));
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// f(0), f(1), ..., f(N - 1), each index a constant (a body this long is past what the compiler unrolls)
template <int... I, typename F>
__device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F&& f) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) { each_of(std::make_integer_sequence<int, N>{}, f); }

// The products where whole rows of x fit a wave's registers (contractions of 256 and 512, no bias) and the output is a large one.
// A wave keeps 32 rows of x as fragments and the weight goes by in LDS, 32 columns and the whole contraction a stage.  A workgroup is eight
// waves, 256 rows; it takes a run of pieces of (256 rows, 64 columns), rows by rows: its ring of stages never empties, and x is read once, or
// twice where a tile is two workgroups'.
//   What bounds hstu_gemm_kernel at a short contraction is that a tile's products and its epilogue take turns (74 k x 512 -> 2048: 139 us
// and 55).  Here the products of a column block stand beside the activation of the one before it, four outputs' steps at a time, and a
// second wave of the SIMD beside both.  74 k x 512 -> 2048 with SiLU 197 -> 150 us, with the pre-activation 216 -> 181, plain 177 -> 142;
// 74 k x 256 -> 1024 74 -> 51, 90 -> 65; added to other rows, 78 k x 512 -> 512 75 -> 66, 25.6 k x 512 -> 2048 98 -> 68.  What is left is the
// matrix pipes' clock on real operands beside the bytes that move: without loads of the weight 11 % less, without stores 14 %, without
// either 25 %.  Two blocks of 32 rows a wave, one wave per SIMD, halve the reads of LDS and are no faster (161, 191, 149; 55, 67).
//   NORM: the layer norm in front of the product on the rows in their registers.  A launch less, and the normed rows are neither written nor
// read again; the norm's 21 instructions for two elements stand before a tile's first product, so that it takes two thirds of what it
// saves (norm and product 78 k x 512 -> 2048 209 -> 200 us, 150 k 385 -> 354, 33 k 96 -> 93, 66 k x 256 -> 1024 72 -> 62, 100 k 93 -> 90; 13 k
// x 512 -> 2048, where more of it is before a first product, 51 -> 55).  (A gate, and the sum of the output product, beside it do not fit the
// registers: 110 -> 250 us.)
//   ALONG: the input's gradient, x w^T, whose weight lies along the contraction: a stage is 32 of its rows, read as they lie.  78 k x 512 by
// 512 60 -> 57 us, 100 k 78 -> 63, 131 k 85 -> 75, 49 k x 256 by 512 25 -> 22,
// and where the rule begins with 512 of depth, 49 k x 512 by 256, 24 -> 24.
template <int K, int OUT, bool NORM, bool ALONG>
__global__ __launch_bounds__(512, 2) void hstu_gemm_rows_kernel(const GemmParams g) {
  constexpr int NS = K / 16, STAGE = K * 64, STAGES = 3, AHEAD = 3;
  constexpr int LP = STAGE / 8192;                       // direct loads of 1 KB per wave and stage
  constexpr bool PRE = OUT == OUT_PRE_SILU, ADD = OUT == OUT_ADD;
  constexpr int STORES = PRE ? 8 : 4, FROM = ADD ? 4 : 0;      // FROM: the product of a step at which its loads begin
  static_assert(LP <= 4, "a step's stores follow its loads");
  static_assert(!ALONG || (OUT == OUT_PLAIN && !NORM), "the input's gradient is a product alone");
  static_assert(NS % (AHEAD + 1) == 0 && 32 % NS == 0 && NS >= 16, "fragments keep their registers from step to step");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const uint32_t smem_lds = __builtin_amdgcn_groupstaticsize();
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5;

  // this workgroup's run of pairs of column blocks, XCD by XCD
  const int pairs = g.cols >> 6;
  const int64_t all = (int64_t)g.row_tiles * pairs;
  const int64_t me = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int64_t first = all * me / gridDim.x, last = all * (me + 1) / gridDim.x;
  if (first >= last) return;
  // (scalars, which a division leaves in vector registers)
  int rt = __builtin_amdgcn_readfirstlane((int)(first / pairs)), pc = __builtin_amdgcn_readfirstlane((int)(first - (int64_t)rt * pairs));
  int todo = __builtin_amdgcn_readfirstlane((int)(last - first));

  // ---- the weight's stages: 32 of its columns in rows of 64 bytes, piece i of a wave 16 rows.  ALONG: 32 of its rows, which lie along the
  // contraction, 16-byte chunk c of row r at c ^ r % 16 (16 rows reach all banks); one slab.
  int sl = __builtin_amdgcn_readfirstlane(64 * pc / g.slab), sc = 64 * pc - sl * g.slab;      // slab and column of the next stage to load
  int wr = 64 * pc;                                      // ALONG: and its row
  constexpr int RC = K / 8;                              // chunks of such a row
  uint32_t po[LP];
#pragma unroll
  for (int i = 0; i < LP; ++i) {
    const int piece = LP * w + i, row = (64 * piece + lane) / RC;
    po[i] = ALONG ? (uint32_t)(row * (int)g.p_stride + 8 * ((lane % RC) ^ (row & 15))) * 2u
                  : (uint32_t)((16 * piece + (lane >> 2)) * (int)g.p_stride + 8 * (lane & 3)) * 2u;
  }
  const char* p_base;
  auto next_columns = [&]() __attribute__((always_inline)) {
    if constexpr (ALONG) {
      p_base = scalar_ptr(g.p[0] + (int64_t)wr * g.p_stride);
      wr = wr + 32 == g.cols ? 0 : wr + 32;
      return;
    }
    p_base = scalar_ptr(g.p[sl] + sc);
    sc += 32;
    if (sc == g.slab) {
      sc = 0;
      sl = (sl + 1) * g.slab == g.cols ? 0 : sl + 1;
    }
  };
  auto dma = [&](int st, int i) __attribute__((always_inline)) {
    lds_dma16(p_base, po[i], smem_lds + (uint32_t)st * STAGE + 1024u * (LP * w + i));
  };

  const int gi = lane & 15;
  const uint32_t at_lane = (uint32_t)((8 * hh + (gi >> 2)) * 64 + 32 * ((lane >> 4) & 1) + 8 * (gi & 3));
  bf16x8 f[AHEAD + 1];
  const uint32_t along_row = (uint32_t)(l32 * 2 * K), along_at = (uint32_t)((hh ^ (l32 & 15)) * 16);
  auto ask = [&](int st, int s) __attribute__((always_inline)) {
    if constexpr (ALONG) {
      f[s % (AHEAD + 1)] = *(const bf16x8*)(smem + st * STAGE + along_row + (along_at ^ (uint32_t)(32 * (s & 7))) + 256 * (s >> 3));
      return;
    }
    const unsigned char* at = smem + st * STAGE + at_lane + 1024 * s;
    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(at));
    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(at + 256));
    struct { short4v a, b; } both = {lo, hi};
    f[s % (AHEAD + 1)] = __builtin_bit_cast(bf16x8, both);
  };

  bf16x8 qf[NS];
  auto load_rows = [&](int tile) __attribute__((always_inline)) {
    int row = 256 * tile + 32 * w + l32;
    row = row < g.rows ? row : g.rows - 1;              // (what a row past the end gives is not stored)
    const bf16_t* at = g.q + (int64_t)row * g.q_stride + 8 * hh;
#pragma unroll
    for (int s = 0; s < NS; ++s) qf[s] = *(const bf16x8*)(at + 16 * s);
  };
  // (waited for here: left to their first use, the waits would stand in the loop and be for every younger load and store in each round)
  auto rows_here = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < NS; ++s) asm volatile("" : "+v"(qf[s]));
  };
  // NORM: the rows' layer norm, as hstu_norm_gate has it (the mean, then the squares about it).  A lane holds half of its row.
  auto both_halves = [&](float x) __attribute__((always_inline)) { return x + __shfl_xor(x, 32, 64); };
  auto norm_rows = [&]() __attribute__((always_inline)) {
    float sum[4] = {0.f, 0.f, 0.f, 0.f}, ss[4] = {0.f, 0.f, 0.f, 0.f};
    // (each pass unpacks the rows again: kept from one to the next they would be two registers for each of theirs)
    each<NS>([&](auto s_) __attribute__((always_inline)) {
      constexpr int s = decltype(s_)::value;
      float x[8];
      unpack8(__builtin_bit_cast(uint4, qf[s]), x);
#pragma unroll
      for (int i = 0; i < 8; ++i) sum[i & 3] += x[i];
      if constexpr (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    });
    rows_here();
    const float mean = both_halves((sum[0] + sum[1]) + (sum[2] + sum[3])) * (1.0f / K);
    each<NS>([&](auto s_) __attribute__((always_inline)) {
      constexpr int s = decltype(s_)::value;
      float x[8];
      unpack8(__builtin_bit_cast(uint4, qf[s]), x);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float d = x[i] - mean;
        ss[i & 3] = __builtin_fmaf(d, d, ss[i & 3]);
      }
      if constexpr (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    });
    rows_here();
    const float rstd = __builtin_amdgcn_rsqf(both_halves((ss[0] + ss[1]) + (ss[2] + ss[3])) * (1.0f / K) + g.eps);
    each<NS>([&](auto s_) __attribute__((always_inline)) {
      constexpr int s = decltype(s_)::value;
      float x[8], ga[8], be[8];
      unpack8(__builtin_bit_cast(uint4, qf[s]), x);
      unpack8(*(const uint4*)(g.gamma + 16 * s + 8 * hh), ga);
      unpack8(*(const uint4*)(g.beta + 16 * s + 8 * hh), be);
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = __builtin_fmaf((x[i] - mean) * rstd, ga[i], be[i]);
      qf[s] = __builtin_bit_cast(bf16x8, pack8(x));
      if constexpr (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    });
    rows_here();
  };

  // ---- the epilogue: 32 rows x 64 columns through the wave's own LDS, rows of 128 bytes, 8-byte piece c of row r at c ^ (r / 2 % 16)
  // (written a column piece of all rows at a time, read a row at a time: all banks both ways)
  // ADD: in fp32, rows of 256 bytes, 16-byte piece c of row r at c ^ r % 16: what is added comes by rows too, and one rounding follows.
  unsigned char* const out_lds = smem + STAGES * STAGE + w * (ADD ? 8192 : 4096);
  unsigned char* const pre_lds = out_lds + 32768;
  float z[4], e[4];
  uint32_t zw[2], ow[2];
  const int wslot = (l32 >> 1) & 15;
  auto put = [&](unsigned char* to, int par, int q4, const uint32_t (&v)[2]) __attribute__((always_inline)) {
    *(uint2*)(to + l32 * 128 + (((8 * par + 2 * q4 + hh) ^ wslot) * 8)) = uint2{v[0], v[1]};
  };
  // part `ph` of 32: eight for each four columns of a lane
  auto epilogue = [&](const floatx16& old, auto par_, auto ph_) __attribute__((always_inline)) {
    constexpr int ph = decltype(ph_)::value, q4 = ph >> 3, par = decltype(par_)::value;
    constexpr bool act = OUT == OUT_SILU || PRE;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr ((ph & 7) == 0) z[i] = old[4 * q4 + i];
      if constexpr ((ph & 7) == 1 && act) e[i] = -1.4426950408889634f * z[i];
      if constexpr ((ph & 7) == 2 && act) e[i] = __builtin_amdgcn_exp2f(e[i]);
      if constexpr ((ph & 7) == 3 && act) e[i] = 1.0f + e[i];
      if constexpr ((ph & 7) == 4 && act) e[i] = __builtin_amdgcn_rcpf(e[i]);
      if constexpr ((ph & 7) == 5 && act) z[i] = z[i] * e[i];
    }
    if constexpr (PRE && (ph & 7) == 0) {
      // (the activation of the stored value, which is what its gradient is taken at)
      zw[0] = pack2(z[0], z[1]);
      zw[1] = pack2(z[2], z[3]);
      z[0] = __builtin_bit_cast(float, zw[0] << 16);
      z[1] = __builtin_bit_cast(float, zw[0] & 0xffff0000u);
      z[2] = __builtin_bit_cast(float, zw[1] << 16);
      z[3] = __builtin_bit_cast(float, zw[1] & 0xffff0000u);
    }
    if constexpr (PRE && (ph & 7) == 4) put(pre_lds, par, q4, zw);
    if constexpr (ADD && (ph & 7) == 7) *(float4*)(out_lds + l32 * 256 + (((8 * par + 2 * q4 + hh) ^ (l32 & 15)) * 16)) = float4{z[0], z[1], z[2], z[3]};
    if constexpr (!ADD && (ph & 7) == 6) {
      ow[0] = pack2(z[0], z[1]);
      ow[1] = pack2(z[2], z[3]);
    }
    if constexpr (!ADD && (ph & 7) == 7) put(out_lds, par, q4, ow);
  };
  typedef uint32_t words __attribute__((ext_vector_type(4)));
  words rows_out[4], rows_pre[4];
  const bool halves = (lane >> 4) & 1;                  // (of 16 bytes, in the other order)
  auto take = [&](const unsigned char* from, int i) __attribute__((always_inline)) {
    const int row = (lane >> 3) + 8 * i;
    const words v = *(const words*)(from + row * 128 + (((lane & 7) ^ ((row >> 2) & 7)) * 16));
    return words{halves ? v[2] : v[0], halves ? v[3] : v[1], halves ? v[0] : v[2], halves ? v[1] : v[3]};
  };
  words add_rows[4];
  auto take_added = [&](int i) __attribute__((always_inline)) {
    const int row = (lane >> 3) + 8 * i;
    const float4 v0 = *(const float4*)(out_lds + row * 256 + (((2 * (lane & 7)) ^ (row & 15)) * 16));
    const float4 v1 = *(const float4*)(out_lds + row * 256 + (((2 * (lane & 7) + 1) ^ (row & 15)) * 16));
    float x[8];
    unpack8(__builtin_bit_cast(uint4, add_rows[i]), x);
    x[0] += v0.x; x[1] += v0.y; x[2] += v0.z; x[3] += v0.w;
    x[4] += v1.x; x[5] += v1.y; x[6] += v1.z; x[7] += v1.w;
    return __builtin_bit_cast(words, pack8(x));
  };
  const uint32_t out_at = (uint32_t)((32 * w + (lane >> 3)) * (int)g.out_stride + 8 * (lane & 7)) * 2u;
  const uint32_t out_step = (uint32_t)(8 * (int)g.out_stride) * 2u;
  // (past the L2s, see store_past; rows past the output's end lie past the buffer's: nothing is stored, and as many stores are under way)
  bf16_t *to_out = g.out[0], *to_pre = g.pre;
  const bf16_t* from_c = g.c;
  uint32_t to_bytes = 0, c_bytes = 0;
  const uint32_t c_at = ADD ? (uint32_t)((32 * w + (lane >> 3)) * (int)g.c_stride + 8 * (lane & 7)) * 2u : 0u;
  const uint32_t c_step = ADD ? (uint32_t)(8 * (int)g.c_stride) * 2u : 0u;
  auto ask_added = [&](int i) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)from_c, 0, (int)c_bytes, 0x00020000);
    add_rows[i] = __builtin_bit_cast(words, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(c_at + i * c_step), 0, 0));
  };
  auto store = [&](bf16_t* base, const words& v, int i) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(base, 0, (int)to_bytes, 0x00020000);
    __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)(out_at + i * out_step), 0, 2);
  };

  const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  floatx16 acc_a = zero, acc_b = zero;
  // One step: the products of a column block, the epilogue of the one before it, the stage after next on its way; in a pair's second step
  // the rows of the pair before are stored.
  auto step = [&](auto par_, int st, floatx16& acc, const floatx16& old) __attribute__((always_inline)) {
    constexpr int par = decltype(par_)::value;
    const int refill = st + 2 >= STAGES ? st + 2 - STAGES : st + 2, next = st + 1 >= STAGES ? 0 : st + 1;
    next_columns();
    each<NS>([&](auto s_) __attribute__((always_inline)) {
      constexpr int s = decltype(s_)::value, PER = 32 / NS;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (s == NS - AHEAD) {
        // (everything asked of the stage is here, and behind the barrier everyone's is: its place can be refilled.  Younger than the next
        // stage's loads: those of the one after it, one pair's stores, and of what is added that pair's rows)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        HSTU_WAIT_VMCNT(LP + STORES + (ADD && par == 0 ? 4 : 0));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if constexpr (s + AHEAD < NS) ask(st, s + AHEAD);
      else ask(next, s + AHEAD - NS);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[s % (AHEAD + 1)], qf[s], s == 0 ? zero : acc, 0, 0, 0);
      if constexpr (ADD && par == 0 && s < 4) ask_added(s);
      if constexpr (s >= FROM && s < FROM + LP) dma(refill, s - FROM);
      if constexpr (par == 1) {
        // (the first part that writes there again is the fifth; of what is added the eighth)
        each<PER>([&](auto i_) __attribute__((always_inline)) {
          constexpr int i = s * PER + decltype(i_)::value;
          if constexpr (i < 4) {
            rows_out[i] = ADD ? take_added(i) : take(out_lds, i);
            if constexpr (PRE) rows_pre[i] = take(pre_lds, i);
          }
        });
        if constexpr (s >= FROM + 4 && s < FROM + 8) {
          store(to_out, rows_out[s - FROM - 4], s - FROM - 4);
          if constexpr (PRE) store(to_pre, rows_pre[s - FROM - 4], s - FROM - 4);
        }
      }
      each<PER>([&](auto i_) __attribute__((always_inline)) {
        epilogue(old, std::integral_constant<int, 1 - par>{}, std::integral_constant<int, s * PER + decltype(i_)::value>{});
      });
    });
    __builtin_amdgcn_sched_barrier(0);
  };

  next_columns();
#pragma unroll
  for (int i = 0; i < LP; ++i) dma(0, i);
  next_columns();
#pragma unroll
  for (int i = 0; i < LP; ++i) dma(1, i);
  load_rows(rt);
  __builtin_amdgcn_sched_barrier(0);
  HSTU_WAIT_VMCNT(LP + NS);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) ask(0, s);
  rows_here();
  int st = 0, have = rt;
  bool as_stored = NORM;
  for (; todo > 0; --todo) {
    if (rt != have) {
      load_rows(rt);
      rows_here();
      have = rt;
      as_stored = NORM;
    }
    if constexpr (NORM) {
      if (as_stored) norm_rows();
      as_stored = false;
    }
    step(std::integral_constant<int, 0>{}, st, acc_a, acc_b);
    st = st + 1 >= STAGES ? 0 : st + 1;
    step(std::integral_constant<int, 1>{}, st, acc_b, acc_a);
    st = st + 1 >= STAGES ? 0 : st + 1;
    const int m0 = 256 * rt;
    const int64_t left = ((int64_t)(g.rows - m0 < 256 ? g.rows - m0 : 256) - 1) * g.out_stride + (g.cols - 64 * pc);
    to_out = g.out[0] + (int64_t)m0 * g.out_stride + 64 * pc;
    to_pre = PRE ? g.pre + (int64_t)m0 * g.out_stride + 64 * pc : nullptr;
    to_bytes = (uint32_t)(left * 2);
    if constexpr (ADD) {
      from_c = g.c + (int64_t)m0 * g.c_stride + 64 * pc;
      c_bytes = (uint32_t)((((int64_t)(g.rows - m0 < 256 ? g.rows - m0 : 256) - 1) * g.c_stride + (g.cols - 64 * pc)) * 2);
    }
    if (++pc == pairs) {
      pc = 0;
      ++rt;
    }
  }
  each<32>([&](auto ph_) __attribute__((always_inline)) {
    epilogue(acc_b, std::integral_constant<int, 1>{}, ph_);
    __builtin_amdgcn_sched_barrier(0);
  });
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (ADD) ask_added(i);
    store(to_out, ADD ? take_added(i) : take(out_lds, i), i);
    if (PRE) store(to_pre, take(pre_lds, i), i);
  }
  HSTU_WAIT_VMCNT(0);        // (no direct load may arrive in LDS that is another workgroup's by then)
}

// A plain product of a short contraction into wide rows (the head of a narrow model), which takes the time of the output's bytes and the
// weight's.  A workgroup stays over a run of pieces of (64 rows, 128 columns), columns by columns: the weight's columns are fragments in registers
// for as long as the run stays in them, a wave's 32 rows of x come one piece ahead, and the only barriers stand where the columns change, so
// that one wave's stores go beside another's products.  (The tiles of hstu_gemm_kernel each begin with loads and end with stores: 1600 x K ->
// 20000 took 22 us at K = 8 too, where a fill of that output takes 11.)
//   1600 x 64 -> 20000 23.3 -> 18.2 us (3.5 TB/s; without the whole lines, see `back`, 20.0), 25600 rows 257 -> 209 (4.9), 400 11.0 -> 10.8,
// 50 10.6 -> 5.0; 50 x 64 -> 131072 43 -> 8.8, 200 x 64 -> 50000 51 -> 12.7; 1600 x 32 -> 20000 20.7 -> 15.6, x 128 29.9 -> 25.8.
template <int K, bool PAST>
__global__ __launch_bounds__(256, K > 64 ? 2 : 4) void hstu_gemm_short_kernel(const GemmParams g) {
  constexpr int NS = K / 16, W_BYTES = 5 * 64 * K;
  __shared__ __attribute__((aligned(16))) unsigned char smem[W_BYTES + 4 * 4096];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hh = lane >> 5, half = w & 1, side = w >> 1;
  const int steps = g.row_tiles;                         // of 64 rows
  // Wave pairs take every second row each: rows whose stride is an odd number of half lines (the example's 20000) begin in the middle of a
  // line by turns, and those are stored from 32 columns further left, so that whole lines are written all the same.
  const int back = ((((uintptr_t)g.out[0] >> 6) & 1) + side * ((g.out_stride >> 5) & 1)) & 1 && g.out_stride % 32 == 0 ? 1 : 0;
  const int64_t all = (int64_t)steps * g.col_tiles;
  const int64_t me = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);     // XCD by XCD
  const int64_t first = all * me / gridDim.x, last = all * (me + 1) / gridDim.x;
  if (first >= last) return;
  int cg = __builtin_amdgcn_readfirstlane((int)(first / steps)), at = __builtin_amdgcn_readfirstlane((int)(first - (int64_t)cg * steps));
  int todo = __builtin_amdgcn_readfirstlane((int)(last - first));

  // the weight's 128 columns and the 32 to their left as blocks of 32, in rows of 64 bytes (as hstu_gemm_rows_kernel has them)
  const int gi = lane & 15;
  const uint32_t at_lane = (uint32_t)((8 * hh + (gi >> 2)) * 64 + 32 * ((lane >> 4) & 1) + 8 * (gi & 3));
  bf16x8 f[2][NS];
  auto columns = [&]() __attribute__((always_inline)) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (20 * K + 255) / 256; ++i) {
      const int piece = 256 * i + tid, block = piece / (4 * K), k = piece / 4 % K, col = 128 * cg - 32 + 32 * block + 8 * (piece & 3);
      uint4 v = {0, 0, 0, 0};
      if (piece >= 20 * K) break;
      if (col >= 0 && col < g.cols) v = *(const uint4*)(g.p[0] + (int64_t)k * g.p_stride + col);
      *(uint4*)(smem + piece * 16) = v;
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const unsigned char* from = smem + (2 * half + b + 1 - back) * (K * 64) + at_lane + 1024 * s;
        const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(from));
        const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(from + 256));
        struct { short4v a, b; } both = {lo, hi};
        f[b][s] = __builtin_bit_cast(bf16x8, both);
      }
  };
  bf16x8 q[NS];
  auto load_rows = [&](int step) __attribute__((always_inline)) {
    int row = 64 * step + 2 * l32 + side;
    row = row < g.rows ? row : g.rows - 1;              // (what a row past the end gives is not stored)
    const bf16_t* from = g.q + (int64_t)row * g.q_stride + 8 * hh;
#pragma unroll
    for (int s = 0; s < NS; ++s) q[s] = *(const bf16x8*)(from + 16 * s);
  };
  // (waited for behind the stores, which are younger: left to their first use in the next round the wait would be for those too)
  auto rows_here = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < NS; ++s) asm volatile("" : "+v"(q[s]));
  };

  // a wave's 32 x 64 results: through its own LDS, as in hstu_gemm_rows_kernel, to whole rows of 128 bytes
  unsigned char* const own = smem + W_BYTES + w * 4096;
  const int wslot = (l32 >> 1) & 15;
  const bool halves = (lane >> 4) & 1;
  typedef uint32_t words __attribute__((ext_vector_type(4)));
  const uint32_t out_at = (uint32_t)((lane >> 3) * 2 * (int)g.out_stride + 8 * (lane & 7)) * 2u, out_step = (uint32_t)(16 * (int)g.out_stride) * 2u;
  const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  load_rows(at);
  columns();
  rows_here();
  for (; todo > 0; --todo) {
    floatx16 acc[2] = {zero, zero};
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[b][s], q[s], acc[b], 0, 0, 0);
    const int m0 = 64 * at + side, n0 = 128 * cg + 64 * half - 32 * back;
    const bool turn = at + 1 == steps;
    at = turn ? 0 : at + 1;
    load_rows(at);
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        *(uint2*)(own + l32 * 128 + (((8 * b + 2 * q4 + hh) ^ wslot) * 8)) = uint2{pack2(acc[b][4 * q4], acc[b][4 * q4 + 1]), pack2(acc[b][4 * q4 + 2], acc[b][4 * q4 + 3])};
    __builtin_amdgcn_wave_barrier();
    // (rows and columns past the output's end lie past the buffer's)
    const int rows_left = (g.rows - m0 + 1) >> 1;
    const int64_t bytes = rows_left > 0 ? (((int64_t)(rows_left < 32 ? rows_left : 32) - 1) * 2 * g.out_stride + (g.cols - n0)) * 2 : 0;
    const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(g.out[0] + (int64_t)m0 * g.out_stride + n0, 0, bytes > 0 ? (int)bytes : 0, 0x00020000);
    const int col = n0 + 8 * (lane & 7);
    const bool inside = col >= 0 && col < g.cols;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = (lane >> 3) + 8 * i;
      const words v = *(const words*)(own + row * 128 + (((lane & 7) ^ ((row >> 2) & 7)) * 16));
      const words o = {halves ? v[2] : v[0], halves ? v[3] : v[1], halves ? v[0] : v[2], halves ? v[1] : v[3]};
      __builtin_amdgcn_raw_buffer_store_b128(o, to, (int)(inside ? out_at + i * out_step : 0x7ffffff0u), 0, PAST ? 2 : 0);
    }
    __builtin_amdgcn_wave_barrier();
    rows_here();
    if (turn && todo > 1) {
      ++cg;
      columns();
    }
  }
}

// Sums the partial products of a split contraction in the order of the splits and rounds them once.
__global__ __launch_bounds__(256) void hstu_gemm_reduce(const GemmParams g) {
  const int64_t per = (int64_t)g.rows * g.cols;
  const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (e >= per) return;
  float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < g.splits; ++s) {
    const float4 a = *(const float4*)(g.partial + s * per + e), b = *(const float4*)(g.partial + s * per + e + 4);
    x[0] += a.x; x[1] += a.y; x[2] += a.z; x[3] += a.w;
    x[4] += b.x; x[5] += b.y; x[6] += b.z; x[7] += b.w;
  }
  const int m = (int)(e / g.cols), n = (int)(e - (int64_t)m * g.cols), sl = n / g.out_slab;
  bf16_t* o = (sl == 0 ? g.out[0] : sl == 1 ? g.out[1] : sl == 2 ? g.out[2] : g.out[3]) + (int64_t)m * g.out_stride + (n - sl * g.out_slab);
  *(uint4*)o = pack8(x);
}

template <int MB, int NB, int WN, bool Q_T, bool P_T, int STAGES, bool UNIFORM, int OUT, bool PAST>
int launch_inst(const GemmParams& g, unsigned blocks, int smem, hipStream_t st) {
  static int granted[64];
  if (int rc = block_allow_lds((const void*)hstu_gemm_kernel<MB, NB, WN, Q_T, P_T, STAGES, UNIFORM, OUT, PAST>, smem, granted)) return rc;
  hipLaunchKernelGGL((hstu_gemm_kernel<MB, NB, WN, Q_T, P_T, STAGES, UNIFORM, OUT, PAST>), dim3(blocks), dim3(128 * WN), smem, st, g);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "gemm kernel launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

template <int MB, int NB, int WN, bool Q_T, bool P_T, int STAGES, bool UNIFORM, int OUT>
int launch_out(const GemmParams& g, unsigned blocks, int smem, hipStream_t st) {
  // (weight gradients are smaller, and 64 x 64 tiles are for products that are)
  if constexpr (!Q_T && MB >= 2) {
    if (store_past(g.rows, g.cols, g.out_stride)) return launch_inst<MB, NB, WN, Q_T, P_T, STAGES, UNIFORM, OUT, true>(g, blocks, smem, st);
  }
  return launch_inst<MB, NB, WN, Q_T, P_T, STAGES, UNIFORM, OUT, false>(g, blocks, smem, st);
}

template <int MB, int NB, int WN, bool Q_T, bool P_T, int STAGES, bool UNIFORM>
int launch_as(const GemmParams& g, unsigned blocks, int smem, hipStream_t st) {
  if constexpr (Q_T) {
    if (g.partial) return launch_out<MB, NB, WN, Q_T, P_T, STAGES, UNIFORM, OUT_PARTIAL>(g, blocks, smem, st);
  } else if constexpr (P_T) {
    if constexpr (UNIFORM) {
      if (!g.c && !g.pre && g.activation) return launch_out<MB, NB, WN, Q_T, P_T, STAGES, UNIFORM, OUT_SILU>(g, blocks, smem, st);
      if (!g.c && g.pre && g.activation) return launch_out<MB, NB, WN, Q_T, P_T, STAGES, UNIFORM, OUT_PRE_SILU>(g, blocks, smem, st);
      if (g.c && !g.pre && !g.activation) return launch_out<MB, NB, WN, Q_T, P_T, STAGES, UNIFORM, OUT_ADD>(g, blocks, smem, st);
    }
    if (g.c || g.pre || g.activation) return launch_out<MB, NB, WN, Q_T, P_T, STAGES, UNIFORM, OUT_ANY>(g, blocks, smem, st);
  }
  return launch_out<MB, NB, WN, Q_T, P_T, STAGES, UNIFORM, OUT_PLAIN>(g, blocks, smem, st);
}

// One slab per tile (per stage, along the contraction); lane offsets within 32 bits.
bool uniform(const GemmParams& g, bool p_t, int tm, int tn) {
  const bool one_slab = p_t ? (g.slab >= g.cols || g.slab % tn == 0) : g.slab % GEMM_BK == 0;
  const int64_t widest = (int64_t)(tm > tn ? tm : tn) * (g.q_stride > g.p_stride ? g.q_stride : g.p_stride) * 2;
  return one_slab && widest < (1LL << 31);
}

template <int MB, int NB, int WN, bool Q_T, bool P_T, int STAGES = 3>
int launch(const GemmParams& p, hipStream_t st) {
  constexpr int TM = 64 * MB, TN = 32 * NB * WN;
  constexpr int ring = STAGES * (TM + TN) * GEMM_BK * 2, out = 2 * WN * 32 * (32 * NB * 4 + 16);
  constexpr int smem = ring > out ? ring : out;
  GemmParams g = p;
  g.row_tiles = (g.rows + TM - 1) / TM;
  g.col_tiles = (g.cols + TN - 1) / TN;
  const int64_t tiles = (int64_t)g.row_tiles * g.col_tiles;
  const int64_t blocks = g.splits >= 8 ? 8LL * ((g.splits + 7) / 8) * tiles
                         : g.splits > 1 ? 8LL * ((tiles * g.splits + 7) / 8) : 8LL * ((g.row_tiles + 7) / 8) * g.col_tiles;
  if (blocks > 0x7fffffffLL) return block_fail(HSTU_BLOCK_ERR_SHAPE, "grid too large");
  if (uniform(g, P_T, TM, TN)) return launch_as<MB, NB, WN, Q_T, P_T, STAGES, true>(g, (unsigned)blocks, smem, st);
  if constexpr (WN == 4) return launch<4, 2, 2, Q_T, P_T>(p, st);
  else return launch_as<MB, NB, WN, Q_T, P_T, STAGES, false>(g, (unsigned)blocks, smem, st);
}

template <bool Q_T, bool P_T>
int launch_sized(const GemmParams& p, hipStream_t st, int tile) {
  if (tile == 3) return launch<4, 2, 4, Q_T, P_T>(p, st);
  if (tile == 2) return launch<4, 2, 2, Q_T, P_T>(p, st);
  if (tile == 1) return launch<2, 2, 2, Q_T, P_T>(p, st);
  return launch<1, 1, 2, Q_T, P_T>(p, st);
}

int64_t tiles_of(int64_t rows, int64_t cols, int tm, int tn) { return ((rows + tm - 1) / tm) * ((cols + tn - 1) / tn); }

// What a product of `tiles` tiles over a contraction of `depth` takes, in microseconds: the CUs run side by side, and one that has n
// workgroups to run needs n times their share of its pipes, but no less than one workgroup by itself takes from its first load to
// its last store.  The constants are a fit to widths of 64 to 2048 and 400 to 131 k rows, every product with every tile: the choice
// by them takes 1.2 % more than the best of the four at each size (the lines by tile counts before it: 12 %).
constexpr int GEMM_TILES = 4;
struct TileCost { int rows, cols; double alone, alone_k, share, share_k, added; };    // added: with an operand that is added to the product
constexpr TileCost TILE_COST[GEMM_TILES] = {
    {64, 64, 4.3, 0.0061, 0.7, 0.0043, 0.1},        // most workgroups: few rows
    {128, 128, 5.8, 0.0102, 2.6, 0.0089, 0.5},      // three workgroups per CU: 6400 x 1024 -> 1024 24 us (256 x 128: 28, 64 x 64: 33)
    {256, 128, 7.7, 0.0146, 4.8, 0.0150, 1.0},      // two: 19200 x 512 -> 2048 61 us (256 x 256: 64, 128 x 128: 64)
    {256, 256, 0.0, 0.0, 7.7, 0.0210, 6.0},         // one: 74 k x 512 -> 2048 194 us (256 x 128: 204), 74 k x 2048 -> 2048 558 (628)
};
double tile_cost(int t, int64_t rows, int64_t cols, double depth, int splits, bool add) {
  const TileCost& c = TILE_COST[t];
  const double n = (double)((tiles_of(rows, cols, c.rows, c.cols) * splits + 255) / 256);
  const double alone = c.alone + c.alone_k * depth, share = n * (c.share + c.share_k * depth + (add ? c.added : 0.0));
  return alone > share ? alone : share;
}

int pick_tile(int64_t rows, int64_t cols, int64_t depth, bool widest, bool add) {
  int best = 0;
  for (int t = 1; t < (widest ? GEMM_TILES : GEMM_TILES - 1); ++t)
    if (tile_cost(t, rows, cols, (double)depth, 1, add) < tile_cost(best, rows, cols, (double)depth, 1, add)) best = t;
  return best;
}

// Tile and splits of a weight gradient, whose contraction is the batch's rows: a split's partial sums are written, read and added (a
// launch, 0.155 us a megabyte, 0.24 a split).  Powers of two, so that whole XCDs share a split; at least 128 rows each.  With
// every (tile, splits) of the sweep timed the choice takes 1.8 % more than the best (the lines before it 36 %: they took eight
// splits where two or none do; 1600 rows, 1024 -> 4096: 62 -> 23 us).
int pick_splits(int64_t rows, int64_t cols, int64_t depth, int* tile) {
  int splits = 1;
  double least = 1e300;
  for (int s = 1; s <= 64 && (s == 1 || depth / s >= 128); s *= 2)
    for (int t = 0; t < GEMM_TILES; ++t) {
      double c = tile_cost(t, rows, cols, (double)depth / s, s, false);
      if (s > 1) c += 2.4 + 0.155 * 8e-6 * s * (double)rows * (double)cols + 0.24 * s;
      if (c < least) { least = c; splits = s; *tile = t; }
    }
  return splits;
}

// Whether hstu_gemm_rows_kernel takes the product: from six pieces for each of its workgroups on.  Below, reading the rows before the first
// product (12 us, twice where a workgroup's run crosses a tile's end) costs more than is won.  us here / with the tiles, at 6.2 pieces:
// 12800 x 512 -> 2048 40.5 / 40.7, with the pre-activation 44 / 49, added to rows 43 / 50, 51200 x 512 -> 512 40 / 42 and 44 / 51, 51200 x 256
// -> 512 25 / 30 and 29 / 35, 25600 x 256 -> 1024 24 / 29; at 12.5: 25600 x 512 -> 2048 62 / 80; at 3.1: 6400 x 512 -> 2048 31 / 24, 25600 x 256 -> 512 19 / 18.
constexpr int ROWS_GRID = 256;                 // a workgroup per CU
bool rows_product(const GemmParams& g) {
  return (g.depth == 256 || g.depth == 512) && !g.bias && (!g.c || (!g.activation && !g.pre && g.c_stride < 1 << 20)) && (g.activation || !g.pre) && g.cols % 64 == 0 && g.slab % 32 == 0 &&
         g.out_stride < 1 << 20 && g.p_stride < 1 << 20 && (int64_t)((g.rows + 255) / 256) * (g.cols / 64) >= 6 * ROWS_GRID;
}

// Whether hstu_gemm_short_kernel takes the product: with rows this wide it does not lose at any number of them (1 to 25600).  Narrower ones
// change their columns too often or leave too few of them: 800 x 64 -> 10000 10.2 us with it and 10.7 with the tiles, x 128 13.9 and 13.0;
// 3200 x 64 -> 5008 14.9 and 13.4, 65536 x 64 -> 1024 38 and 35, x 128 52 and 41.  Rows that are no whole half lines are stored in parts of lines
// here: with few rows alone (250 x 64 -> 16392 8.4 and 9.7, 500 10.5 and 9.9, 25600 362 and 262; 800 x 64 -> 50000 27 and 31).
bool short_product(const GemmParams& g) {
  return (g.depth == 32 || g.depth == 64 || g.depth == 128) && !g.bias && !g.c && !g.activation && !g.pre && g.cols >= 16384 && g.slab == g.cols &&
         (g.out_stride % 32 == 0 || g.rows <= (g.cols >= 32768 ? 1024 : 256)) && g.out_stride < 1 << 20 && g.p_stride < 1 << 20;
}

template <int K>
int launch_short(GemmParams g, hipStream_t st) {
  g.row_tiles = (g.rows + 63) / 64;
  g.col_tiles = (g.cols + 32 + 127) / 128;              // (rows that are stored from 32 columns further left)
  const dim3 grid(256 * (K > 64 ? 2 : 4));
  if (store_past(g.rows, g.cols, g.out_stride)) hipLaunchKernelGGL((hstu_gemm_short_kernel<K, true>), grid, dim3(256), 0, st, g);
  else hipLaunchKernelGGL((hstu_gemm_short_kernel<K, false>), grid, dim3(256), 0, st, g);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "gemm kernel launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

template <int K, int OUT, bool NORM = false, bool ALONG = false>
int launch_rows_as(GemmParams g, hipStream_t st) {
  static int granted[64];
  constexpr int smem = 3 * K * 64 + (OUT == OUT_PRE_SILU || OUT == OUT_ADD ? 65536 : 32768);
  g.row_tiles = (g.rows + 255) / 256;
  if (int rc = block_allow_lds((const void*)hstu_gemm_rows_kernel<K, OUT, NORM, ALONG>, smem, granted)) return rc;
  hipLaunchKernelGGL((hstu_gemm_rows_kernel<K, OUT, NORM, ALONG>), dim3(ROWS_GRID), dim3(512), smem, st, g);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "gemm kernel launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}
template <int K>
int launch_rows(const GemmParams& g, bool along, hipStream_t st) {
  if (along) return launch_rows_as<K, OUT_PLAIN, false, true>(g, st);
  if (g.gamma) return launch_rows_as<K, OUT_SILU, true>(g, st);
  if (g.c) return launch_rows_as<K, OUT_ADD>(g, st);
  if (g.pre) return launch_rows_as<K, OUT_PRE_SILU>(g, st);
  if (g.activation) return launch_rows_as<K, OUT_SILU>(g, st);
  return launch_rows_as<K, OUT_PLAIN>(g, st);
}

// out = act(x w + c + bias) for widths that the kernel above cannot fetch 16 bytes at a time: element by element, fp32 products.  (One
// workgroup per 64 x 64 outputs, 16 of the contraction at a time through LDS, 4 x 4 outputs per thread.)
struct PlainParams {
  const bf16_t *x, *w, *bias, *c;
  bf16_t* out;
  int64_t x_stride, c_stride;
  int32_t M, N, K, activation, col_tiles;
};
__global__ __launch_bounds__(256) void hstu_gemm_plain(const PlainParams p) {
  __shared__ float xs[16][65], ws[16][65];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int m0 = (int)(blockIdx.x / p.col_tiles) * 64, n0 = (int)(blockIdx.x % p.col_tiles) * 64;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < p.K; k0 += 16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = tid + 256 * i;
      const int xr = e >> 4, xk = e & 15, wk = e >> 6, wc = e & 63;
      xs[xk][xr] = m0 + xr < p.M && k0 + xk < p.K ? (float)p.x[(int64_t)(m0 + xr) * p.x_stride + k0 + xk] : 0.f;
      ws[wk][wc] = n0 + wc < p.N && k0 + wk < p.K ? (float)p.w[(int64_t)(k0 + wk) * p.N + n0 + wc] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 16; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(xs[k][ty + 16 * i], ws[k][tx + 16 * j], acc[i][j]);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = m0 + ty + 16 * i, n = n0 + tx + 16 * j;
      if (m < p.M && n < p.N) {
        float v = acc[i][j];
        if (p.c) v += (float)p.c[(int64_t)m * p.c_stride + n];
        if (p.bias) v += (float)p.bias[n];
        p.out[(int64_t)m * p.N + n] = (bf16_t)(p.activation ? silu(v) : v);
      }
    }
}

}  // namespace

extern "C" {

// (nothing is needed; callers that ask are given a size they can allocate)
size_t hstu_gemm_silu_workspace_bytes(void) { return 256; }

int hstu_gemm_silu_fwd(const HstuGemmSiluArgs* a, void* stream) {
  HstuGemmSiluArgs own;
  a = block_today(a, own, sizeof(HstuGemmSiluArgs), sizeof(HstuGemmSiluArgs));
  if (!a) return block_fail(HSTU_BLOCK_ERR_NULL, "args is null");
  if (a->struct_size != sizeof(HstuGemmSiluArgs) || a->version != HSTU_BLOCK_ABI_VERSION)
    return block_fail(HSTU_BLOCK_ERR_VERSION, "gemm args struct_size/version (%u/%u) do not match this library (%zu/%d)",
                      a->struct_size, a->version, sizeof(HstuGemmSiluArgs), HSTU_BLOCK_ABI_VERSION);
  if (a->M < 0 || a->N < 1 || a->K < 1 || a->M > 0x7fffffffLL || a->x_stride < a->K)
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "bad shape M=%lld N=%d K=%d x_stride=%lld", (long long)a->M, a->N, a->K, (long long)a->x_stride);
  if (a->activation != 0 && a->activation != 1) return block_fail(HSTU_BLOCK_ERR_SHAPE, "activation must be 0 (none) or 1 (silu)");
  block_clear_error();
  if (a->M == 0) return HSTU_BLOCK_OK;
  if (!a->x || !a->w || !a->out) return block_fail(HSTU_BLOCK_ERR_NULL, "x, w and out must be non-null");
  if (!block_aligned16(a->x) || !block_aligned16(a->w) || !block_aligned16(a->out) || !block_aligned16(a->bias) || !block_aligned16(a->workspace) || (a->x_stride & 7))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "x, w, out, bias and workspace must be 16-byte aligned and x_stride a multiple of 8 elements");
  if (a->c && (!block_aligned16(a->c) || (a->c_stride & 7) || a->c_stride < a->N))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "c must be 16-byte aligned with a row stride that is a multiple of 8 elements and >= N");
  if (a->workspace_bytes && !a->workspace) return block_fail(HSTU_BLOCK_ERR_WORKSPACE, "workspace_bytes without a workspace");
  constexpr int64_t PART = 1 << 28;              // rows of a launch: 32-bit indices
  for (int64_t m0 = 0; m0 < a->M; m0 += PART) {
    const int64_t rows = a->M - m0 < PART ? a->M - m0 : PART;
    const bf16_t* x = (const bf16_t*)a->x + m0 * a->x_stride;
    const bf16_t* c = a->c ? (const bf16_t*)a->c + m0 * a->c_stride : nullptr;
    bf16_t* out = (bf16_t*)a->out + m0 * a->N;
    if (a->N % 8 == 0 && a->K % 8 == 0) {
      HstuGemmArgs g;
      memset(&g, 0, sizeof(g));
      g.struct_size = sizeof(g); g.version = HSTU_BLOCK_ABI_VERSION;
      g.op = HSTU_GEMM_NN; g.activation = a->activation;
      g.M = rows; g.N = a->N; g.K = a->K; g.slabs = 1;
      g.x = x; g.x_stride = a->x_stride; g.w[0] = const_cast<void*>(a->w); g.bias = a->bias; g.c = c; g.c_stride = a->c_stride; g.out = out;
      if (int rc = hstu_gemm(&g, stream)) return rc;
      continue;
    }
    PlainParams p = {x, (const bf16_t*)a->w, (const bf16_t*)a->bias, c, out, a->x_stride, a->c_stride, (int32_t)rows, a->N, a->K, a->activation, 0};
    p.col_tiles = (a->N + 63) / 64;
    const int64_t blocks = (rows + 63) / 64 * p.col_tiles;
    if (blocks > 0x7fffffffLL) return block_fail(HSTU_BLOCK_ERR_SHAPE, "grid too large");
    hipLaunchKernelGGL(hstu_gemm_plain, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "gemm kernel launch: %s", hipGetErrorString(e));
  }
  return HSTU_BLOCK_OK;
}

size_t hstu_gemm_workspace_bytes(int32_t op, int64_t M, int32_t N, int32_t K) {
  if (op != HSTU_GEMM_TN || M < 1 || N < 1 || K < 1) return 0;
  int tile;
  const int s = pick_splits(K, N, M, &tile);
  return s > 1 ? (size_t)s * (size_t)K * (size_t)N * sizeof(float) : 0;
}

int hstu_gemm(const HstuGemmArgs* a, void* stream) {
  HstuGemmArgs own;
  a = block_today(a, own, 0, sizeof(HstuGemmArgs));
  if (!a) return block_fail(HSTU_BLOCK_ERR_NULL, "args is null");
  if (a->struct_size != sizeof(HstuGemmArgs) || a->version != HSTU_BLOCK_ABI_VERSION)
    return block_fail(HSTU_BLOCK_ERR_VERSION, "gemm args struct_size/version (%u/%u) do not match this library (%zu/%d)",
                      a->struct_size, a->version, sizeof(HstuGemmArgs), HSTU_BLOCK_ABI_VERSION);
  if (a->op < HSTU_GEMM_NN || a->op > HSTU_GEMM_TN) return block_fail(HSTU_BLOCK_ERR_SHAPE, "unknown op %d", a->op);
  if (a->M < 0 || a->M > 0x3fffffff || a->N < 8 || a->K < 8 || (a->N & 7) || (a->K & 7) || a->slabs < 1 || a->slabs > HSTU_GEMM_MAX_SLABS ||
      a->N % a->slabs || (a->N / a->slabs & 7))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "N, K and the slabs must be multiples of 8: got M=%lld N=%d K=%d in %d slabs", (long long)a->M, a->N, a->K,
                      a->slabs);
  const int slab = a->N / a->slabs;
  const bool tn = a->op == HSTU_GEMM_TN;
  if ((a->x_stride & 7) || a->x_stride < (a->op == HSTU_GEMM_NT ? a->N : a->K))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "x_stride must be a multiple of 8 and cover a row, got %lld", (long long)a->x_stride);
  if (a->M == 0 && !tn) return HSTU_BLOCK_OK;
  bool ok = block_aligned16(a->x) && block_aligned16(a->bias) && block_aligned16(a->c) && block_aligned16(a->pre) && (a->x || a->M == 0);
  for (int i = 0; i < a->slabs; ++i) ok = ok && a->w[i] && block_aligned16(a->w[i]);
  if (tn) ok = ok && (a->y || a->M == 0) && block_aligned16(a->y) && (a->y_stride & 7) == 0 && a->y_stride >= a->N;
  else ok = ok && a->out && block_aligned16(a->out) && (!a->c || ((a->c_stride & 7) == 0 && a->c_stride >= a->N));
  if (!ok) return block_fail(HSTU_BLOCK_ERR_SHAPE, "operands must be present, 16-byte aligned, with row strides of whole 16-byte pieces");
  if (a->op != HSTU_GEMM_NN && (a->bias || a->c || a->pre || a->activation))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "bias, c, pre and the activation belong to the forward product");
  hipStream_t st = (hipStream_t)stream;
  GemmParams p = {};
  p.q = (const bf16_t*)a->x;
  p.q_stride = a->x_stride;
  p.splits = 1;
  p.slab = slab;
  p.bias = (const bf16_t*)a->bias; p.c = (const bf16_t*)a->c; p.c_stride = a->c_stride;
  p.pre = (bf16_t*)a->pre;
  p.activation = a->activation;
  if (tn) {
    p.rows = a->K; p.cols = a->N; p.depth = (int32_t)a->M;
    p.p[0] = (const bf16_t*)a->y; p.p_stride = a->y_stride;
    p.slab = a->N;                       // y is one matrix; the slabs are the output's
    p.out_slab = slab;
    for (int i = 0; i < a->slabs; ++i) p.out[i] = (bf16_t*)const_cast<void*>(a->w[i]);
    p.out_stride = slab;
    int tile;
    p.splits = pick_splits(a->K, a->N, a->M, &tile);
    p.depth_per_split = p.depth;
    if (p.splits == 1) return launch_sized<true, true>(p, st, tile);
    const size_t need = hstu_gemm_workspace_bytes(a->op, a->M, a->N, a->K);
    if (!a->workspace || a->workspace_bytes < need || !block_aligned16(a->workspace))
      return block_fail(HSTU_BLOCK_ERR_WORKSPACE, "workspace of %zu bytes needed (hstu_gemm_workspace_bytes), got %zu", need,
                        a->workspace ? a->workspace_bytes : (size_t)0);
    p.partial = (float*)a->workspace;
    const int per = ((p.depth + p.splits - 1) / p.splits + GEMM_BK - 1) / GEMM_BK * GEMM_BK;
    p.depth_per_split = per;
    if (int rc = launch_sized<true, true>(p, st, tile)) return rc;
    const int64_t n8 = (int64_t)p.rows * p.cols / 8;
    hipLaunchKernelGGL(hstu_gemm_reduce, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, st, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "gemm reduction launch: %s", hipGetErrorString(e));
    return HSTU_BLOCK_OK;
  }
  // (one slab may be narrower than a stage, several may not: the kernel moves on by at most one per stage)
  if (a->op == HSTU_GEMM_NT && a->slabs > 1 && slab < GEMM_BK)
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "slabs of at least %d columns are needed here, got %d", GEMM_BK, slab);
  for (int i = 0; i < HSTU_GEMM_MAX_SLABS; ++i) p.p[i] = (const bf16_t*)a->w[i < a->slabs ? i : a->slabs - 1];
  p.p_stride = slab;
  p.rows = (int32_t)a->M;
  p.out[0] = (bf16_t*)a->out;
  if (a->op == HSTU_GEMM_NN) {
    p.cols = p.out_slab = a->N;
    p.out_stride = a->N;
    p.depth = p.depth_per_split = a->K;
    if (rows_product(p)) return p.depth == 512 ? launch_rows<512>(p, false, st) : launch_rows<256>(p, false, st);
    if (short_product(p)) return p.depth == 128 ? launch_short<128>(p, st) : p.depth == 64 ? launch_short<64>(p, st) : launch_short<32>(p, st);
    return launch_sized<false, true>(p, st, pick_tile(p.rows, p.cols, p.depth, uniform(p, true, 256, 256), p.c != nullptr));
  }
  p.cols = p.out_slab = a->K;
  p.out_stride = a->K;
  p.depth = p.depth_per_split = a->N;
  if (a->slabs == 1 && rows_product(p)) return p.depth == 512 ? launch_rows<512>(p, true, st) : launch_rows<256>(p, true, st);
  return launch_sized<false, false>(p, st, pick_tile(p.rows, p.cols, p.depth, uniform(p, false, 256, 256), false));
}

// (from sixteen pieces a workgroup on: see NORM)
int hstu_norm_gemm_takes(int64_t M, int32_t N, int32_t K, int32_t slabs) {
  if (M < 1 || M > 0x3fffffff || N < 64 || slabs < 1 || slabs > HSTU_GEMM_MAX_SLABS || N % slabs) return 0;
  GemmParams p = {};
  p.rows = (int32_t)M; p.cols = N; p.depth = K; p.slab = p.p_stride = N / slabs; p.out_stride = N;
  p.activation = 1;
  return rows_product(p) && (int64_t)((p.rows + 255) / 256) * (N / 64) >= 16 * ROWS_GRID ? 1 : 0;
}

int hstu_norm_gemm(const HstuNormGemmArgs* a, void* stream) {
  if (!a) return block_fail(HSTU_BLOCK_ERR_NULL, "args is null");
  if (a->struct_size != sizeof(HstuNormGemmArgs) || a->version != HSTU_BLOCK_ABI_VERSION)
    return block_fail(HSTU_BLOCK_ERR_VERSION, "norm-gemm args struct_size/version (%u/%u) do not match this library (%zu/%d)", a->struct_size, a->version,
                      sizeof(HstuNormGemmArgs), HSTU_BLOCK_ABI_VERSION);
  if (!hstu_norm_gemm_takes(a->M, a->N, a->K, a->slabs))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "no kernel for M=%lld N=%d K=%d in %d slabs (hstu_norm_gemm_takes)", (long long)a->M, a->N, a->K, a->slabs);
  bool ok = a->x && a->gamma && a->beta && a->out && a->x_stride >= a->K && (a->x_stride & 7) == 0;
  for (const void* t : {a->x, a->gamma, a->beta, (const void*)a->out}) ok = ok && block_aligned16(t);
  for (int i = 0; i < a->slabs; ++i) ok = ok && a->w[i] && block_aligned16(a->w[i]);
  if (!ok) return block_fail(HSTU_BLOCK_ERR_SHAPE, "operands must be present, 16-byte aligned, with row strides of whole 16-byte pieces");
  block_clear_error();
  GemmParams p = {};
  p.q = (const bf16_t*)a->x; p.q_stride = a->x_stride;
  p.gamma = (const bf16_t*)a->gamma; p.beta = (const bf16_t*)a->beta;
  p.eps = a->eps;
  p.splits = 1;
  p.slab = a->N / a->slabs;
  for (int i = 0; i < HSTU_GEMM_MAX_SLABS; ++i) p.p[i] = (const bf16_t*)a->w[i < a->slabs ? i : a->slabs - 1];
  p.p_stride = p.slab;
  p.rows = (int32_t)a->M; p.cols = p.out_slab = a->N; p.out_stride = a->N;
  p.depth = p.depth_per_split = a->K;
  p.out[0] = (bf16_t*)a->out;
  p.activation = 1;
  return a->K == 512 ? launch_rows<512>(p, false, (hipStream_t)stream) : launch_rows<256>(p, false, (hipStream_t)stream);
}

}  // extern "C"
