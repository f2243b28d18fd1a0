// Whole HSTU blocks in one launch, for short sequences and narrow models in inference (recml/layers/keras/hstu.py:442-474): layer
// norm, the U, Q, K and V projections with SiLU, causal pointwise attention, layer norm times gate, output projection, residual.
//
// One workgroup per sequence of up to 64 positions, at head dims of 16 and widths of 32 and 64: everything between the first block's
// input and the last one's output stays in LDS (107 KB a block, 150 with the next one's parameters).  What bounds such a block is none of
// its work (2 MFLOP and 45 KB a sequence) but its launches, and in one launch the vector instructions and the LDS latencies of seven
// phases on a CU of its own.  Four blocks of 32 sequences of 50 at width 64 take 72 us as five launches each, 32.4 as one launch each
// and 22.7 as one for all of them; 512 sequences 142 / 70 / 47.  (Sixteen waves in place of eight: 22.8 / 47.8.)  Of the 32.4 the
// attention's blocks had half, at 130 instructions each: keys read by transpose, the mask on the diagonal only and the table in LDS
// leave 50.  Every value that the separate kernels round to bf16 on its way through memory is rounded here, and none else: the weights
// of the attention stay in fp32, as the kernels for head dims of 16 have them.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "hstu_block.h"
#include "hstu_block_common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4v* lds_short4_ptr;

constexpr int HD = 16;           // head dim
constexpr int ROWS = 64;         // positions of a workgroup
constexpr int WAVES = 8;         // two to a head at width 64: each step is a chain of a few hundred cycles per block, so more waves, not fewer
constexpr int THREADS = 64 * WAVES;
constexpr float SMALL_LOG2E = 1.4426950408889634f;

constexpr int MOST = HSTU_BLOCK_SMALL_STACK;      // blocks of a launch (their parameters are kernel arguments: 120 bytes each)

struct SmallWeights {
  const bf16_t *in_gamma, *in_beta, *attn_gamma, *attn_beta, *w[4], *wb[4], *w_out, *b_out;
  float eps;
};

struct SmallParams {
  const bf16_t* tokens;
  bf16_t* out;
  const int32_t* seq_lens;       // or null: L
  const int32_t* seq_offsets;    // or null: sequence b at row b L, all L rows of it computed
  const float* pos_tab;
  const bf16_t *end_gamma, *end_beta;      // a layer norm behind the last block, or null
  int32_t L, pos_heads, n;
  float end_eps, alpha, inv_n;
  SmallWeights blk[MOST];
};

template <int W>
struct SmallShape {
  static constexpr int ROW = W * 2 + 16;           // bytes of a row of W values in LDS (16 more: other banks)
  static constexpr int ROW4 = 8 * W + 16;          // of a projection's 4 W
  static constexpr int X = 0;                      // tokens, as they come                          [64][ROW]
  static constexpr int N = X + ROWS * ROW;         // normed; later the attention's result          [64][ROW]
  static constexpr int G = N + ROWS * ROW;         // gated                                         [64][ROW]
  static constexpr int P = G + ROWS * ROW;         // u, q, k, v                                    [64][ROW4]
  static constexpr int TAB = P + ROWS * ROW4;      // the position table's entries for key - query = 1 - ROWS .. 0, a row per head (padded: the
                                                   // pairs of a block on the diagonal above it read on)   [W / HD][TAB_ROW] fp32
  static constexpr int TAB_ROW = ROWS + 16;
  static constexpr int BLK = TAB + W / HD * TAB_ROW * 4;      // a block's parameters; with several blocks twice, taken in turn
  static constexpr int WQ = 0;                     //   the projections' weight                     [W][ROW4]
  static constexpr int WO = WQ + W * ROW4;         //   the output's                                [W][ROW]
  static constexpr int V = WO + W * ROW;           //   nine vectors: norms' scales and offsets, the projections' and the output's biases (or zeros)
  static constexpr int PARAMS = V + 9 * 2 * W;
  static constexpr int lds(int n) { return BLK + (n > 1 ? 2 : 1) * PARAMS; }
};

enum { V_IN_GAMMA, V_IN_BETA, V_ATTN_GAMMA, V_ATTN_BETA, V_BIAS, V_OUT_BIAS = V_BIAS + 4 };

// A block's parameters on their way from memory to LDS: asked for while the block before is worked on
template <int W>
struct SmallFetch {
  static constexpr int CPR = W / 8;                // 16-byte pieces of a row
  static constexpr int N = (5 * W * CPR + THREADS - 1) / THREADS;
  typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
  uintx4 v[N], x;
  __device__ __forceinline__ void ask(const SmallWeights& p, int tid) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = tid + THREADS * i, m = e / (W * CPR), r = (e / CPR) % W, c = e % CPR;
      if (m < 5) {
        const bf16_t* w = m == 0 ? p.w[0] : m == 1 ? p.w[1] : m == 2 ? p.w[2] : m == 3 ? p.w[3] : p.w_out;
        v[i] = *(const uintx4*)(w + r * W + 8 * c);
      }
    }
    if (tid < 9 * CPR) {
      const int i = tid / CPR, c = tid % CPR;
      const bf16_t* src = i == V_IN_GAMMA ? p.in_gamma : i == V_IN_BETA ? p.in_beta : i == V_ATTN_GAMMA ? p.attn_gamma : i == V_ATTN_BETA ? p.attn_beta
                          : i == V_BIAS ? p.wb[0] : i == V_BIAS + 1 ? p.wb[1] : i == V_BIAS + 2 ? p.wb[2] : i == V_BIAS + 3 ? p.wb[3] : p.b_out;
      x = uintx4{0u, 0u, 0u, 0u};
      if (src) x = *(const uintx4*)(src + 8 * c);
    }
  }
  __device__ __forceinline__ void put(unsigned char* to, int tid) const {
    using S = SmallShape<W>;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = tid + THREADS * i, m = e / (W * CPR), r = (e / CPR) % W, c = e % CPR;
      if (m < 5) *(uintx4*)(m < 4 ? to + S::WQ + r * S::ROW4 + 2 * W * m + 16 * c : to + S::WO + r * S::ROW + 16 * c) = v[i];
    }
    if (tid < 9 * CPR) *(uintx4*)(to + S::V + 2 * W * (tid / CPR) + 16 * (tid % CPR)) = x;
  }
};

// the sum over aligned groups of N lanes (4 or 8), by additions whose operand is moved on the way
template <int N>
__device__ __forceinline__ float near_sum(float v) {
  auto moved = [](float x, auto ctrl) __attribute__((always_inline)) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  v += moved(v, std::integral_constant<int, 0xB1>{});            // the neighbour
  v += moved(v, std::integral_constant<int, 0x4E>{});            // the pair beside it
  if constexpr (N == 8) v += moved(v, std::integral_constant<int, 0x141>{});      // the other four of eight
  return v;
}

// Layer norm of rows of W values: W / 8 lanes a row, eight values each; y = gate * (gamma (x - mean) rstd + beta)
template <int W, bool GATE>
__device__ __forceinline__ void norm_rows(const unsigned char* in, unsigned char* out, const unsigned char* gate, const bf16_t* gamma, const bf16_t* beta,
                                          float eps, int tid) {
  constexpr int LPR = W / 8;
  if (tid >= ROWS * LPR) return;
  const int row = tid / LPR, at = 8 * (tid % LPR);
  float x[8], g[8], b[8], u[8], y[8];
  unpack8(*(const uint4*)(in + row * SmallShape<W>::ROW + 2 * at), x);
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) sum += x[e];
  const float mean = near_sum<LPR>(sum) / (float)W;
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float d = x[e] - mean;
    ss += d * d;
  }
  const float rstd = __builtin_amdgcn_rsqf(near_sum<LPR>(ss) / (float)W + eps);
  unpack8(*(const uint4*)(gamma + at), g);
  unpack8(*(const uint4*)(beta + at), b);
  if constexpr (GATE) unpack8(*(const uint4*)(gate + row * SmallShape<W>::ROW4 + 2 * at), u);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    y[e] = __builtin_fmaf((x[e] - mean) * rstd, g[e], b[e]);
    if constexpr (GATE) y[e] *= u[e];
  }
  *(uint4*)(out + row * SmallShape<W>::ROW + 2 * at) = pack8(y);
}

// NB 32 x 32 blocks of x w, `step` columns apart, transposed: lane (l32, hh), register 4 g + t: row r0 + l32, column n0 + 8 g + 4 hh + t.
// x: rows of ROW bytes; w: rows (along the contraction) of `pitch` bytes.  All operands are asked for ahead of the first product: one by
// one each waits for LDS by itself.
template <int W, int NB>
__device__ __forceinline__ void products(floatx16 (&acc)[NB], const unsigned char* x, int r0, const unsigned char* w, int pitch, int n0, int step, int lane) {
  const int l32 = lane & 31, hh = lane >> 5, gi = lane & 15;
  bf16x8 b[W / 16];
  struct Two { short4v a, b; } f[W / 16][NB];
  // (16 lanes name four rows of 16 columns and get a column of them each)
  const unsigned char* const wr = w + (8 * hh + (gi >> 2)) * pitch + 2 * (n0 + 16 * ((lane >> 4) & 1) + 4 * (gi & 3));
#pragma unroll
  for (int s = 0; s < W / 16; ++s) {
    b[s] = *(const bf16x8*)(x + (r0 + l32) * SmallShape<W>::ROW + 32 * s + 16 * hh);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const unsigned char* const at = wr + 16 * s * pitch + 2 * step * i;
      f[s][i] = Two{__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)at), __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(at + 4 * pitch))};
    }
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < W / 16; ++s)
#pragma unroll
    for (int i = 0; i < NB; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, f[s][i]), b[s], acc[i], 0, 0, 0);
}

template <int W>
__global__ __launch_bounds__(THREADS, W == 64 ? 2 : 6) void hstu_block_small(const SmallParams p) {       // (waves per SIMD that the LDS has room for)
  using S = SmallShape<W>;
  extern __shared__ __attribute__((aligned(16))) unsigned char sm[];
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  int64_t row0;
  int n, rows;                     // valid positions; rows to compute
  if (p.seq_offsets) {
    const int o0 = p.seq_offsets[b];
    n = p.seq_offsets[b + 1] - o0;
    n = n < 0 ? 0 : (n < p.L ? n : p.L);
    rows = n;
    row0 = o0;
  } else {
    row0 = (int64_t)b * p.L;
    rows = p.L;
    n = rows;
    if (p.seq_lens) {
      n = p.seq_lens[b];
      n = n < 0 ? 0 : (n < p.L ? n : p.L);
    }
  }
  if (rows == 0) return;

  // ---- everything from memory
  constexpr int CPR = W / 8;       // 16-byte pieces of a row
  SmallFetch<W> next;
  next.ask(p.blk[0], tid);
#pragma unroll
  for (int i = 0; i < (ROWS * CPR + THREADS - 1) / THREADS; ++i) {
    const int e = tid + THREADS * i, r = e / CPR, c = e % CPR;
    if (r < ROWS) {
      const uint4 v = *(const uint4*)(p.tokens + (row0 + (r < rows ? r : rows - 1)) * W + 8 * c);    // (rows past the end repeat the last: not stored)
      *(uint4*)(sm + S::X + r * S::ROW + 16 * c) = v;
    }
  }
  next.put(sm + S::BLK, tid);
  if (p.pos_tab) {
    for (int e = tid; e < p.pos_heads * S::TAB_ROW; e += THREADS) {
      const int h = e / S::TAB_ROW, d = e % S::TAB_ROW - (ROWS - 1);
      *(float*)(sm + S::TAB + 4 * e) = d <= 0 && d > -p.L ? p.pos_tab[(int64_t)h * (2 * p.L - 1) + p.L - 1 + d] : 0.f;
    }
  }

  for (int i = 0; i < p.n; ++i) {
    unsigned char* const blk = sm + S::BLK + (i & 1) * S::PARAMS;
    const bf16_t* const vec = (const bf16_t*)(blk + S::V);
    const float eps = p.blk[i].eps;
    const bool biased = p.blk[i].wb[0] != nullptr, out_biased = p.blk[i].b_out != nullptr;
    __syncthreads();                 // x and the parameters are there
    if (i + 1 < p.n) next.ask(p.blk[i + 1], tid);
    norm_rows<W, false>(sm + S::X, sm + S::N, nullptr, vec + V_IN_GAMMA * W, vec + V_IN_BETA * W, eps, tid);
    __syncthreads();

    const int l32 = lane & 31, hh = lane >> 5;
    // ---- u, q, k, v = silu(normed w + bias): 32 rows and NB blocks of 32 columns to a wave
    {
      constexpr int GROUPS = WAVES / 2, COLS = 4 * W / 32, NB = COLS / GROUPS > 0 ? COLS / GROUPS : 1;
      const int r0 = 32 * (wv & 1), n0 = 32 * (wv >> 1);
      if (r0 < rows && (wv >> 1) < COLS) {
        floatx16 acc[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[k][e] = 0.f;
        if (biased) {
#pragma unroll
          for (int k = 0; k < NB; ++k)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
              const uint2 two = *(const uint2*)(vec + V_BIAS * W + n0 + 32 * GROUPS * k + 8 * g + 4 * hh);
              acc[k][4 * g] = __builtin_bit_cast(float, two.x << 16);
              acc[k][4 * g + 1] = __builtin_bit_cast(float, two.x & 0xffff0000u);
              acc[k][4 * g + 2] = __builtin_bit_cast(float, two.y << 16);
              acc[k][4 * g + 3] = __builtin_bit_cast(float, two.y & 0xffff0000u);
            }
        }
        products<W, NB>(acc, sm + S::N, r0, blk + S::WQ, S::ROW4, n0, 32 * GROUPS, lane);
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          const int c0 = n0 + 32 * GROUPS * k;
          const bool live = c0 < 3 * W || r0 + l32 < n;           // (values of keys past the end: zeros, as their weights are)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = silu(acc[k][4 * g + e]);
            const uint2 two = {pack2(x[0], x[1]), pack2(x[2], x[3])};
            *(uint2*)(sm + S::P + (r0 + l32) * S::ROW4 + 2 * (c0 + 8 * g + 4 * hh)) = uint2{live ? two.x : 0u, live ? two.y : 0u};
          }
        }
      }
    }
    __syncthreads();

    // ---- attention: a head to PER waves, 16 queries by 16 keys at a time; S^T = K Q^T by one bf16 product (head dim 16), O^T += V^T P^T
    // by fp32 ones whose k-slot l / 16 of the r-th is key 4 (l / 16) + r: what register r of S^T's lane holds.  Keys past the sequence's
    // end are met by queries past it only, whose rows are zeros; the diagonal is the last block of a query's.
    const int m = lane & 15, g = lane >> 4;
    constexpr int PER = WAVES / (W / HD);          // waves to a head, which take its blocks of queries in turn
    {
      const int h = wv / PER;
      const unsigned char* base = sm + S::P + 2 * HD * h;
      const float* const bias = (const float*)(sm + S::TAB) + (p.pos_heads > 1 ? h : 0) * S::TAB_ROW + ROWS - 1 + 4 * g - m;
      // (16 lanes name four rows of 16 channels and get a channel of them each)
      const unsigned char* const vt = base + 6 * W + (4 * g + (m >> 2)) * S::ROW4 + 8 * (m & 3);
      for (int q0 = 16 * (wv % PER); q0 < rows; q0 += 16 * PER) {
        floatx4 o = {0.f, 0.f, 0.f, 0.f};
        if (q0 < n) {
          const short4v q = *(const short4v*)(base + (q0 + m) * S::ROW4 + 2 * W + 8 * g);
          auto keys = [&](int k0, bool diagonal) __attribute__((always_inline)) {
            const short4v k = *(const short4v*)(base + (k0 + m) * S::ROW4 + 4 * W + 8 * g);
            const short4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(vt + k0 * S::ROW4));
            floatx4 x = {0.f, 0.f, 0.f, 0.f};
            x = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(k, q, x, 0, 0, 0);
            float u[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) u[r] = p.alpha * x[r];
            if (p.pos_tab) {
#pragma unroll
              for (int r = 0; r < 4; ++r) u[r] += bias[k0 - q0 + r];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              u[r] = u[r] * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-u[r] * SMALL_LOG2E));
              if (diagonal) u[r] = 4 * g + r <= m ? u[r] : 0.f;
            }
            const uint2 vb = __builtin_bit_cast(uint2, v);
            const float vf[4] = {__builtin_bit_cast(float, vb.x << 16), __builtin_bit_cast(float, vb.x & 0xffff0000u), __builtin_bit_cast(float, vb.y << 16),
                                 __builtin_bit_cast(float, vb.y & 0xffff0000u)};
#pragma unroll
            for (int r = 0; r < 4; ++r) o = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[r], u[r], o, 0, 0, 0);
          };
          for (int k0 = 0; k0 < q0; k0 += 16) keys(k0, false);
          keys(q0, true);
        }
        // lane (m, g), register r: channel 4 g + r of query m
        const bool in = q0 + m < n;
        *(uint2*)(sm + S::N + (q0 + m) * S::ROW + 2 * HD * h + 8 * g) =
            uint2{in ? pack2(o[0] * p.inv_n, o[1] * p.inv_n) : 0u, in ? pack2(o[2] * p.inv_n, o[3] * p.inv_n) : 0u};
      }
    }
    __syncthreads();
    norm_rows<W, true>(sm + S::N, sm + S::G, sm + S::P, vec + V_ATTN_GAMMA * W, vec + V_ATTN_BETA * W, eps, tid);
    if (i + 1 < p.n) next.put(sm + S::BLK + ((i + 1) & 1) * S::PARAMS, tid);      // (last read two phases into the block before)
    __syncthreads();

    // ---- out = tokens + gated w_out + bias: a 32 x 32 block to a wave, over the tokens that it reads
    for (int t = wv; t < 2 * (W / 32); t += WAVES) {
      const int n0 = 32 * (t >> 1), r0 = 32 * (t & 1);
      if (r0 >= rows) continue;
      const int r = r0 + l32;
      floatx16 acc[1];
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[0][e] = 0.f;
      products<W, 1>(acc, sm + S::G, r0, blk + S::WO, S::ROW, n0, 0, lane);
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int c = n0 + 8 * g4 + 4 * hh;
        uint2* const at = (uint2*)(sm + S::X + r * S::ROW + 2 * c);
        const uint2 res = *at;
        float x[4] = {acc[0][4 * g4] + __builtin_bit_cast(float, res.x << 16), acc[0][4 * g4 + 1] + __builtin_bit_cast(float, res.x & 0xffff0000u),
                      acc[0][4 * g4 + 2] + __builtin_bit_cast(float, res.y << 16), acc[0][4 * g4 + 3] + __builtin_bit_cast(float, res.y & 0xffff0000u)};
        if (out_biased) {
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] += (float)vec[V_OUT_BIAS * W + c + e];
        }
        *at = uint2{pack2(x[0], x[1]), pack2(x[2], x[3])};
      }
    }
  }
  __syncthreads();
  int from = S::X;
  if (p.end_gamma) {
    norm_rows<W, false>(sm + S::X, sm + S::N, nullptr, p.end_gamma, p.end_beta, p.end_eps, tid);
    from = S::N;
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < (ROWS * CPR + THREADS - 1) / THREADS; ++i) {
    const int e = tid + THREADS * i, r = e / CPR, c = e % CPR;
    if (r < rows) *(uint4*)(p.out + (row0 + r) * W + 8 * c) = *(const uint4*)(sm + from + r * S::ROW + 16 * c);
  }
}

template <int W>
int launch_small(const SmallParams& p, int B, hipStream_t st) {
  static int granted[64];
  if (int rc = block_allow_lds((const void*)hstu_block_small<W>, SmallShape<W>::lds(2), granted)) return rc;
  hipLaunchKernelGGL(hstu_block_small<W>, dim3((unsigned)B), dim3(THREADS), SmallShape<W>::lds(p.n), st, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "small block kernel launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

int check_small(const HstuBlockSmallArgs* a, bool first, bool last) {
  if (a->struct_size != sizeof(HstuBlockSmallArgs) || a->version != HSTU_BLOCK_ABI_VERSION)
    return block_fail(HSTU_BLOCK_ERR_VERSION, "small block args struct_size/version (%u/%u) do not match this library (%zu/%d)", a->struct_size,
                      a->version, sizeof(HstuBlockSmallArgs), HSTU_BLOCK_ABI_VERSION);
  if (!hstu_block_small_takes(a->B, a->L, a->heads, a->head_dim, a->width))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "not a small block: B=%d L=%d heads=%d head_dim=%d width=%d", a->B, a->L, a->heads, a->head_dim, a->width);
  block_clear_error();
  bool ok = (a->tokens || !first) && (a->out || !last) && a->in_gamma && a->in_beta && a->attn_gamma && a->attn_beta && a->w_out;
  for (int i = 0; i < 4; ++i) ok = ok && a->w[i] && (!a->w_bias[i] == !a->w_bias[0]);
  if (!ok) return block_fail(HSTU_BLOCK_ERR_NULL, "tokens, out, the norms and the weights must be non-null, the biases all or none");
  const void* const aligned[] = {first ? a->tokens : nullptr, last ? a->out : nullptr, a->in_gamma, a->in_beta, a->attn_gamma, a->attn_beta, a->w[0],
                                 a->w[1], a->w[2], a->w[3], a->w_out, a->w_bias[0], a->w_bias[1], a->w_bias[2], a->w_bias[3], a->b_out};
  for (const void* x : aligned)
    if (!block_aligned16(x)) return block_fail(HSTU_BLOCK_ERR_SHAPE, "tokens, out, norms, weights and biases must be 16-byte aligned");
  if (a->pos_tab && a->pos_heads != 1 && a->pos_heads != a->heads)
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "the position table has %d heads, the block %d", a->pos_heads, a->heads);
  return HSTU_BLOCK_OK;
}

}  // namespace

extern "C" {

// The shapes there are, and of those the ones where this is the faster form.  A workgroup takes the time of 64 positions whatever its
// sequence has, one a CU at width 64 (107 KB of LDS): GPU us a block in five launches / in one, 4 heads: 32 sequences of 50 18.1 / 8.4,
// 512 35.4 / 18.0, 8192 266 / 224; 1024 of 24 35 / 25, but 8192 of 24 137 / 184.
int hstu_block_small_takes(int32_t B, int32_t L, int32_t heads, int32_t head_dim, int32_t width) {
  return head_dim == HD && (width == 32 || width == 64) && heads * head_dim == width && L >= 1 && L <= ROWS && B >= 1 && B <= 65535 && (B <= 1024 || L >= 48);
}

int hstu_block_small_fwd(const HstuBlockSmallArgs* a, void* stream) {
  if (!a) return block_fail(HSTU_BLOCK_ERR_NULL, "args is null");
  return hstu_block_small_stack_fwd(a, 1, nullptr, nullptr, 0.f, stream);
}

int hstu_block_small_stack_fwd(const HstuBlockSmallArgs* a, int32_t n, const void* end_gamma, const void* end_beta, float end_eps, void* stream) {
  if (!a) return block_fail(HSTU_BLOCK_ERR_NULL, "args is null");
  if (n < 1 || n > HSTU_BLOCK_SMALL_STACK) return block_fail(HSTU_BLOCK_ERR_SHAPE, "1 to %d blocks to a call, not %d", HSTU_BLOCK_SMALL_STACK, n);
  SmallParams p = {};
  for (int i = 0; i < n; ++i) {
    const HstuBlockSmallArgs& b = a[i];
    if (int rc = check_small(&b, i == 0, i == n - 1)) return rc;
    if (b.B != a->B || b.L != a->L || b.width != a->width || b.seq_lens != a->seq_lens || b.seq_offsets != a->seq_offsets || b.pos_tab != a->pos_tab ||
        b.pos_heads != a->pos_heads || b.alpha != a->alpha || b.inv_n != a->inv_n)
      return block_fail(HSTU_BLOCK_ERR_SHAPE, "block %d of a call has another batch, width, table or scale than the first", i);
    SmallWeights& w = p.blk[i];
    w.in_gamma = (const bf16_t*)b.in_gamma; w.in_beta = (const bf16_t*)b.in_beta;
    w.attn_gamma = (const bf16_t*)b.attn_gamma; w.attn_beta = (const bf16_t*)b.attn_beta;
    for (int k = 0; k < 4; ++k) { w.w[k] = (const bf16_t*)b.w[k]; w.wb[k] = (const bf16_t*)b.w_bias[k]; }
    w.w_out = (const bf16_t*)b.w_out; w.b_out = (const bf16_t*)b.b_out;
    w.eps = b.eps;
  }
  if (!end_gamma != !end_beta) return block_fail(HSTU_BLOCK_ERR_NULL, "the closing norm takes a scale and an offset, or neither");
  if (!block_aligned16(end_gamma) || !block_aligned16(end_beta)) return block_fail(HSTU_BLOCK_ERR_SHAPE, "the closing norm's scale and offset must be 16-byte aligned");
  p.tokens = (const bf16_t*)a->tokens; p.out = (bf16_t*)a[n - 1].out;
  p.seq_lens = a->seq_lens; p.seq_offsets = a->seq_offsets;
  p.pos_tab = a->pos_tab; p.pos_heads = a->pos_heads;
  p.end_gamma = (const bf16_t*)end_gamma; p.end_beta = (const bf16_t*)end_beta; p.end_eps = end_eps;
  p.L = a->L; p.n = n; p.alpha = a->alpha; p.inv_n = a->inv_n;
  return a->width == 64 ? launch_small<64>(p, a->B, (hipStream_t)stream) : launch_small<32>(p, a->B, (hipStream_t)stream);
}

}  // extern "C"
