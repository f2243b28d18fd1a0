// A whole HSTU block in one launch, for short sequences and narrow models in inference (recml/layers/keras/hstu.py:442-474): layer
// norm, the U, Q, K and V projections with SiLU, causal pointwise attention, layer norm times gate, output projection, residual.
//
// One workgroup per sequence of up to 64 positions, at head dims of 16 and widths of 32 and 64: everything between the block's input
// and its output stays in LDS (95 KB).  What bounds such a block is none of its work (2 MFLOP and 45 KB a sequence) but its launches:
// as five kernels a block of 32 sequences of 50 takes 18.1 us of the GPU and 19 of the host, as this one 8.4 and 8.  Every value that
// those kernels round to bf16 on its way through memory is rounded here, and none else: the weights of the attention stay in fp32, as
// the kernels for head dims of 16 have them.
#include <hip/hip_runtime.h>
#include <stdint.h>

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

struct SmallParams {
  const bf16_t* tokens;
  bf16_t* out;
  const int32_t* seq_lens;       // or null: L
  const int32_t* seq_offsets;    // or null: sequence b at row b L, all L rows of it computed
  const bf16_t *in_gamma, *in_beta, *attn_gamma, *attn_beta, *w[4], *wb[4], *w_out, *b_out;
  const float* pos_tab;
  int32_t L, pos_heads;
  float eps, alpha, inv_n;
};

template <int W>
struct SmallShape {
  static constexpr int ROW = W * 2 + 16;           // bytes of a row of W values in LDS (16 more: other banks)
  static constexpr int ROW4 = 8 * W + 16;          // of a projection's 4 W
  static constexpr int X = 0;                      // tokens, as they come                          [64][ROW]
  static constexpr int N = X + ROWS * ROW;         // normed; later the attention's result          [64][ROW]
  static constexpr int G = N + ROWS * ROW;         // gated                                         [64][ROW]
  static constexpr int P = G + ROWS * ROW;         // u, q, k, v                                    [64][ROW4]
  static constexpr int WQ = P + ROWS * ROW4;       // the projections' weight                       [W][ROW4]
  static constexpr int WO = WQ + W * ROW4;         // the output's                                  [W][ROW]
  static constexpr int V = WO + W * ROW;           // nine vectors: norms' scales and offsets, the projections' and the output's biases (or zeros)
  static constexpr int LDS = V + 9 * 2 * W;
};

enum { V_IN_GAMMA, V_IN_BETA, V_ATTN_GAMMA, V_ATTN_BETA, V_BIAS, V_OUT_BIAS = V_BIAS + 4 };

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
  const float mean = group_sum<LPR>(sum) / (float)W;
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float d = x[e] - mean;
    ss += d * d;
  }
  const float rstd = __builtin_amdgcn_rsqf(group_sum<LPR>(ss) / (float)W + eps);
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

// A 32 x 32 block of x w, transposed: lane (l32, hh), register 4 g + t: row r0 + l32, column n0 + 8 g + 4 hh + t.  x: rows of ROW bytes; w:
// rows (along the contraction) of `pitch` bytes
template <int W>
__device__ __forceinline__ floatx16 product(const unsigned char* x, int r0, const unsigned char* w, int pitch, int n0, int lane) {
  const int l32 = lane & 31, hh = lane >> 5, gi = lane & 15;
  floatx16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
  for (int s = 0; s < W / 16; ++s) {
    const bf16x8 b = *(const bf16x8*)(x + (r0 + l32) * SmallShape<W>::ROW + 32 * s + 16 * hh);
    // (16 lanes name four rows of 16 columns and get a column of them each)
    const unsigned char* at = w + (16 * s + 8 * hh + (gi >> 2)) * pitch + 2 * (n0 + 16 * ((lane >> 4) & 1) + 4 * (gi & 3));
    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)at);
    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_ptr)(at + 4 * pitch));
    struct { short4v a, b; } both = {lo, hi};
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, both), b, acc, 0, 0, 0);
  }
  return acc;
}

__device__ __forceinline__ float bf16_at(const void* p) { return (float)*(const bf16_t*)p; }

template <int W>
__global__ __launch_bounds__(THREADS) void hstu_block_small(const SmallParams p) {
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
#pragma unroll
  for (int i = 0; i < (ROWS * CPR + THREADS - 1) / THREADS; ++i) {
    const int e = tid + THREADS * i, r = e / CPR, c = e % CPR;
    if (r < ROWS) {
      const uint4 v = *(const uint4*)(p.tokens + (row0 + (r < rows ? r : rows - 1)) * W + 8 * c);    // (rows past the end repeat the last: not stored)
      *(uint4*)(sm + S::X + r * S::ROW + 16 * c) = v;
    }
  }
#pragma unroll
  for (int i = 0; i < (5 * W * CPR + THREADS - 1) / THREADS; ++i) {
    const int e = tid + THREADS * i, m = e / (W * CPR), r = (e / CPR) % W, c = e % CPR;
    if (m < 5) {
      const bf16_t* w = m == 0 ? p.w[0] : m == 1 ? p.w[1] : m == 2 ? p.w[2] : m == 3 ? p.w[3] : p.w_out;
      const uint4 v = *(const uint4*)(w + r * W + 8 * c);
      *(uint4*)(m < 4 ? sm + S::WQ + r * S::ROW4 + 2 * W * m + 16 * c : sm + S::WO + r * S::ROW + 16 * c) = v;
    }
  }
  const bf16_t* const vec = (const bf16_t*)(sm + S::V);
  if (tid < 9 * CPR) {
    const int i = tid / CPR, c = tid % CPR;
    const bf16_t* src = i == V_IN_GAMMA ? p.in_gamma : i == V_IN_BETA ? p.in_beta : i == V_ATTN_GAMMA ? p.attn_gamma : i == V_ATTN_BETA ? p.attn_beta
                        : i == V_BIAS ? p.wb[0] : i == V_BIAS + 1 ? p.wb[1] : i == V_BIAS + 2 ? p.wb[2] : i == V_BIAS + 3 ? p.wb[3] : p.b_out;
    uint4 v = {0u, 0u, 0u, 0u};
    if (src) v = *(const uint4*)(src + 8 * c);
    *(uint4*)(sm + S::V + 2 * W * i + 16 * c) = v;
  }
  __syncthreads();
  norm_rows<W, false>(sm + S::X, sm + S::N, nullptr, vec + V_IN_GAMMA * W, vec + V_IN_BETA * W, p.eps, tid);
  __syncthreads();

  const int l32 = lane & 31, hh = lane >> 5;
  // ---- u, q, k, v = silu(normed w + bias): a 32 x 32 block to a wave
  for (int t = wv; t < 2 * (4 * W / 32); t += WAVES) {
    const int n0 = 32 * (t >> 1), r0 = 32 * (t & 1);
    if (r0 < rows) {
      const floatx16 acc = product<W>(sm + S::N, r0, sm + S::WQ, S::ROW4, n0, lane);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = silu(acc[4 * g + e] + (float)vec[V_BIAS * W + n0 + 8 * g + 4 * hh + e]);
        *(uint2*)(sm + S::P + (r0 + l32) * S::ROW4 + 2 * (n0 + 8 * g + 4 * hh)) = uint2{pack2(x[0], x[1]), pack2(x[2], x[3])};
      }
    }
  }
  __syncthreads();

  // ---- attention: a head to PER waves, 16 queries by 16 keys at a time; S^T = K Q^T by one bf16 product (head dim 16), O^T += V^T P^T by fp32 ones
  // whose k-slot l / 16 of the r-th is key 4 (l / 16) + r: what register r of S^T's lane holds
  const int m = lane & 15, g = lane >> 4;
  constexpr int PER = WAVES / (W / HD);          // waves to a head, which take its blocks of queries in turn
  {
    const int h = wv / PER;
    const unsigned char* base = sm + S::P + 2 * HD * h;
    const float* tab = p.pos_tab ? p.pos_tab + (int64_t)(p.pos_heads > 1 ? h : 0) * (2 * p.L - 1) + p.L - 1 : nullptr;
    for (int q0 = 16 * (wv % PER); q0 < rows; q0 += 16 * PER) {
      floatx4 o = {0.f, 0.f, 0.f, 0.f};
      const short4v q = *(const short4v*)(base + (q0 + m) * S::ROW4 + 2 * W + 8 * g);
      const int qi = q0 + m;
      for (int k0 = 0; k0 <= q0 && k0 < n && q0 < n; k0 += 16) {
        const short4v k = *(const short4v*)(base + (k0 + m) * S::ROW4 + 4 * W + 8 * g);
        floatx4 x = {0.f, 0.f, 0.f, 0.f};
        x = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(k, q, x, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = k0 + 4 * g + r;
          const bool keep = j <= qi && qi < n;           // (j <= qi < n)
          float u = p.alpha * x[r];
          if (tab) u += tab[keep ? j - qi : 0];
          x[r] = keep ? u * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-u * SMALL_LOG2E)) : 0.f;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = k0 + 4 * g + r < n - 1 ? k0 + 4 * g + r : n - 1;      // (what stands past the sequence's end is nobody's value)
          o = __builtin_amdgcn_mfma_f32_16x16x4f32(bf16_at(base + j * S::ROW4 + 6 * W + 2 * m), x[r], o, 0, 0, 0);
        }
      }
      // lane (m, g), register r: channel 4 g + r of query m
      *(uint2*)(sm + S::N + (q0 + m) * S::ROW + 2 * HD * h + 8 * g) = uint2{pack2(o[0] * p.inv_n, o[1] * p.inv_n), pack2(o[2] * p.inv_n, o[3] * p.inv_n)};
    }
  }
  __syncthreads();
  norm_rows<W, true>(sm + S::N, sm + S::G, sm + S::P, vec + V_ATTN_GAMMA * W, vec + V_ATTN_BETA * W, p.eps, tid);
  __syncthreads();

  // ---- out = tokens + gated w_out + bias: a 32 x 32 block to a wave
  for (int t = wv; t < 2 * (W / 32); t += WAVES) {
    const int n0 = 32 * (t >> 1), r0 = 32 * (t & 1);
    if (r0 >= rows) continue;
    const floatx16 acc = product<W>(sm + S::G, r0, sm + S::WO, S::ROW, n0, lane);
    const int r = r0 + l32;
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const int c = n0 + 8 * g4 + 4 * hh;
      const uint2 res = *(const uint2*)(sm + S::X + r * S::ROW + 2 * c);
      float x[4] = {acc[4 * g4] + __builtin_bit_cast(float, res.x << 16), acc[4 * g4 + 1] + __builtin_bit_cast(float, res.x & 0xffff0000u),
                    acc[4 * g4 + 2] + __builtin_bit_cast(float, res.y << 16), acc[4 * g4 + 3] + __builtin_bit_cast(float, res.y & 0xffff0000u)};
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] += (float)vec[V_OUT_BIAS * W + c + e];
      if (r < rows) *(uint2*)(p.out + (row0 + r) * W + c) = uint2{pack2(x[0], x[1]), pack2(x[2], x[3])};
    }
  }
}

template <int W>
int launch_small(const SmallParams& p, int B, hipStream_t st) {
  static int granted[64];
  constexpr int smem = SmallShape<W>::LDS;
  if (int rc = block_allow_lds((const void*)hstu_block_small<W>, smem, granted)) return rc;
  hipLaunchKernelGGL(hstu_block_small<W>, dim3((unsigned)B), dim3(THREADS), smem, st, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "small block kernel launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

}  // namespace

extern "C" {

// The shapes there are, and of those the ones where this is the faster form.  A workgroup takes the time of 64 positions whatever its
// sequence has, one a CU at width 64 (95 KB of LDS): GPU us a block in five launches / in one, 4 heads: 32 sequences of 50 18.1 / 8.4,
// 512 35.4 / 18.0, 8192 266 / 224; 1024 of 24 35 / 25, but 8192 of 24 137 / 184.
int hstu_block_small_takes(int32_t B, int32_t L, int32_t heads, int32_t head_dim, int32_t width) {
  return head_dim == HD && (width == 32 || width == 64) && heads * head_dim == width && L >= 1 && L <= ROWS && B >= 1 && B <= 65535 && (B <= 1024 || L >= 48);
}

int hstu_block_small_fwd(const HstuBlockSmallArgs* a, void* stream) {
  if (!a) return block_fail(HSTU_BLOCK_ERR_NULL, "args is null");
  if (a->struct_size != sizeof(HstuBlockSmallArgs) || a->version != HSTU_BLOCK_ABI_VERSION)
    return block_fail(HSTU_BLOCK_ERR_VERSION, "small block args struct_size/version (%u/%u) do not match this library (%zu/%d)", a->struct_size,
                      a->version, sizeof(HstuBlockSmallArgs), HSTU_BLOCK_ABI_VERSION);
  if (!hstu_block_small_takes(a->B, a->L, a->heads, a->head_dim, a->width))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "not a small block: B=%d L=%d heads=%d head_dim=%d width=%d", a->B, a->L, a->heads, a->head_dim, a->width);
  block_clear_error();
  bool ok = a->tokens && a->out && a->in_gamma && a->in_beta && a->attn_gamma && a->attn_beta && a->w_out;
  for (int i = 0; i < 4; ++i) ok = ok && a->w[i] && (!a->w_bias[i] == !a->w_bias[0]);
  if (!ok) return block_fail(HSTU_BLOCK_ERR_NULL, "tokens, out, the norms and the weights must be non-null, the biases all or none");
  const void* const aligned[] = {a->tokens, a->out, a->in_gamma, a->in_beta, a->attn_gamma, a->attn_beta, a->w[0], a->w[1], a->w[2], a->w[3], a->w_out,
                                 a->w_bias[0], a->w_bias[1], a->w_bias[2], a->w_bias[3], a->b_out};
  for (const void* x : aligned)
    if (!block_aligned16(x)) return block_fail(HSTU_BLOCK_ERR_SHAPE, "tokens, out, norms, weights and biases must be 16-byte aligned");
  if (a->pos_tab && a->pos_heads != 1 && a->pos_heads != a->heads)
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "the position table has %d heads, the block %d", a->pos_heads, a->heads);
  SmallParams p = {};
  p.tokens = (const bf16_t*)a->tokens; p.out = (bf16_t*)a->out;
  p.seq_lens = a->seq_lens; p.seq_offsets = a->seq_offsets;
  p.in_gamma = (const bf16_t*)a->in_gamma; p.in_beta = (const bf16_t*)a->in_beta;
  p.attn_gamma = (const bf16_t*)a->attn_gamma; p.attn_beta = (const bf16_t*)a->attn_beta;
  for (int i = 0; i < 4; ++i) { p.w[i] = (const bf16_t*)a->w[i]; p.wb[i] = (const bf16_t*)a->w_bias[i]; }
  p.w_out = (const bf16_t*)a->w_out; p.b_out = (const bf16_t*)a->b_out;
  p.pos_tab = a->pos_tab; p.pos_heads = a->pos_heads;
  p.L = a->L; p.eps = a->eps; p.alpha = a->alpha; p.inv_n = a->inv_n;
  return a->width == 64 ? launch_small<64>(p, a->B, (hipStream_t)stream) : launch_small<32>(p, a->B, (hipStream_t)stream);
}

}  // extern "C"
