// Fused steps of the HSTU block around the attention kernel and of the model's front end, for
// gfx950 (MI355X): see include/hstu_block.h.
//
//   hstu_norm_gate   out = u * layer_norm(attn)   (recml/layers/keras/hstu.py:471-472)
//                    one wavefront per token row, 16 bytes per lane and trip: the row is read once,
//                    kept in registers for the two reductions (mean, then centred sum of squares) and
//                    written once: 3 x width x 2 bytes of HBM traffic per row, which is the bound.
//   hstu_norm_gate_bwd  the gradients of that step (and, without a gate, of a plain layer norm): one
//                    pass over the row, its gradient and the gate; column sums for dgamma / dbeta in
//                    registers, one partial row per workgroup, added in a fixed order by hstu_colsum.
//   hstu_embed_norm  out = layer_norm(scale * table[ids] + pos_table[positions])   (hstu.py:593-601)
//                    the same one-wave-per-row scheme with a gathered row: one read of the table row
//                    (and of the small position table, which stays in cache), one write.

#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <type_traits>

#include "hstu_block.h"
#include "hstu_block_common.h"

namespace {
thread_local char g_err[512] = "";
}

int block_fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

void block_clear_error() { g_err[0] = 0; }

int block_allow_lds(const void* fn, int bytes, int* granted) {
  constexpr int kMaxDev = 64;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "hipGetDevice: %s", hipGetErrorString(e));
  if (dev >= 0 && dev < kMaxDev && __atomic_load_n(&granted[dev], __ATOMIC_ACQUIRE) >= bytes) return HSTU_BLOCK_OK;
  e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "hipFuncSetAttribute(%d bytes of LDS): %s", bytes, hipGetErrorString(e));
  if (dev >= 0 && dev < kMaxDev) __atomic_store_n(&granted[dev], bytes, __ATOMIC_RELEASE);
  return HSTU_BLOCK_OK;
}

namespace {

struct NormGateParams {
  const bf16_t* a;
  const bf16_t* u;
  bf16_t* out;
  const bf16_t* gamma;
  const bf16_t* beta;
  int64_t rows, a_stride, u_stride, out_stride;
  // out is a padded batch [rows / L][L] whose sequence b starts at row seq_offsets[b] of `a`; rows past a sequence's end
  // are zeros (null: row r of `a` is row r of `out`)
  const int32_t* seq_offsets;
  int32_t L;
  int32_t width;
  float eps;
};

// LPR lanes per row (a row of up to 64, 128, 256 elements takes 8, 16, 32 lanes, so that a wavefront holds 8, 4, 2 of them;
// longer ones a whole wavefront); lane l of a row owns its 8-element pieces l, l + LPR, ... (CH of them at most).
template <int CH, int LPR>
__global__ __launch_bounds__(256) void hstu_norm_gate(const NormGateParams p) {
  constexpr int RPW = 64 / LPR;
  const int lane = threadIdx.x & (LPR - 1);
  const int64_t row = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * RPW + ((threadIdx.x & 63) / LPR);
  if (row >= p.rows) return;
  int64_t src = row;
  bf16_t* orow = p.out + row * p.out_stride;
  if (p.seq_offsets) {
    const int b = (int)(row / p.L), i = (int)(row - (int64_t)b * p.L), o0 = p.seq_offsets[b];
    src = o0 + i;
    if (i >= p.seq_offsets[b + 1] - o0) {
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int e = (c * LPR + lane) * 8;
        if (e < p.width) *(uint4*)(orow + e) = uint4{0u, 0u, 0u, 0u};
      }
      return;
    }
  }
  const bf16_t* ar = p.a + src * p.a_stride;
  const bf16_t* ur = p.u ? p.u + row * p.u_stride : nullptr;   // no gate: the plain layer norm
  float x[CH][8];
  float sum = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int e = (c * LPR + lane) * 8;
    if (e < p.width) {
      unpack8(*(const uint4*)(ar + e), x[c]);
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += x[c][i];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[c][i] = 0.f;
    }
  }
  const float mean = group_sum<LPR>(sum) / (float)p.width;
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int e = (c * LPR + lane) * 8;
    if (e < p.width) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float d = x[c][i] - mean;
        ss += d * d;
      }
    }
  }
  const float rstd = __builtin_amdgcn_rsqf(group_sum<LPR>(ss) / (float)p.width + p.eps);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int e = (c * LPR + lane) * 8;
    if (e < p.width) {
      float g[8], b[8], uu[8];
      unpack8(*(const uint4*)(p.gamma + e), g);
      unpack8(*(const uint4*)(p.beta + e), b);
      if (ur) {
        unpack8(*(const uint4*)(ur + e), uu);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) uu[i] = 1.f;
      }
      float y[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = uu[i] * __builtin_fmaf((x[c][i] - mean) * rstd, g[i], b[i]);
      *(uint4*)(orow + e) = pack8(y);
    }
  }
}

struct NormGateBwdParams {
  const bf16_t* a;
  const bf16_t* u;
  const bf16_t* dout;
  const bf16_t* gamma;
  const bf16_t* beta;
  bf16_t* da;
  bf16_t* du;
  float* partial;          // [gridDim.x][2 * width]: each workgroup's sums for dgamma, then for dbeta
  const bf16_t* u_pre;     // u = silu(u_pre), and du is the gradient of u_pre; or null
  const bf16_t* add;       // added to da (the gradient that reaches `a` past the norm); or null
  const int32_t* row_map;  // row r of dout is row row_map[r] of the buffer; or null
  int64_t rows, a_stride, u_stride, dout_stride, da_stride, du_stride, u_pre_stride, add_stride;
  int32_t width;
  float eps;
};

// Backward of out = u * (gamma * xhat + beta), xhat = (a - mean) * rstd, for the gradient g of out:
//   du = g * (gamma * xhat + beta),  gn = g * u  (the gradient at the normalised row; gn = g without a gate)
//   dgamma += gn * xhat,  dbeta += gn           (summed over the rows)
//   da = rstd * (gn gamma - mean_w(gn gamma) - xhat * mean_w(gn gamma xhat))
// Rows on lanes as in the forward, a workgroup walking over rows with the grid's stride: the row,
// its gradient and the gate are read once, da and du written once (5 x width x 2 bytes per row, the
// bound).  The two column sums stay in registers over a wave's rows, are added across the workgroup's
// four waves through LDS and leave as one partial row per workgroup; hstu_colsum adds those in a fixed
// order, so the result does not depend on the timing of the run.
template <int CH, int LPR>
__global__ __launch_bounds__(256) void hstu_norm_gate_bwd(const NormGateBwdParams p) {
  __shared__ float red[4][CH * LPR * 8];
  constexpr int RPW = 64 / LPR;
  const int lane = threadIdx.x & (LPR - 1), w = threadIdx.x >> 6;
  const float inv_w = 1.f / (float)p.width;
  float dg[CH][8], db[CH][8];
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int i = 0; i < 8; ++i) dg[c][i] = db[c][i] = 0.f;
  for (int64_t row = ((int64_t)blockIdx.x * 4 + w) * RPW + ((threadIdx.x & 63) / LPR); row < p.rows; row += (int64_t)gridDim.x * 4 * RPW) {
    const bf16_t* ar = p.a + row * p.a_stride;
    const int64_t grow = p.row_map ? p.row_map[row] : row;
    const bf16_t* gr = p.dout + grow * p.dout_stride;
    float x[CH][8], g[CH][8];
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int e = (c * LPR + lane) * 8;
      if (e < p.width) {
        unpack8(*(const uint4*)(ar + e), x[c]);
        unpack8(*(const uint4*)(gr + e), g[c]);
#pragma unroll
        for (int i = 0; i < 8; ++i) sum += x[c][i];
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) x[c][i] = g[c][i] = 0.f;
      }
    }
    const float mean = group_sum<LPR>(sum) * inv_w;
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int e = (c * LPR + lane) * 8;
      if (e < p.width) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float d = x[c][i] - mean;
          ss += d * d;
        }
      }
    }
    const float rstd = __builtin_amdgcn_rsqf(group_sum<LPR>(ss) * inv_w + p.eps);
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int e = (c * LPR + lane) * 8;
      if (e < p.width) {
        float gm[8];
        unpack8(*(const uint4*)(p.gamma + e), gm);
        if (p.u) {
          float bt[8], uu[8], y[8];
          unpack8(*(const uint4*)(p.beta + e), bt);
          // (the gate itself from u_pre too: 80 of 480 MB not read, 9.5 us less at 78 k rows of 512)
          unpack8(p.u_pre ? *(const uint4*)(p.u_pre + row * p.u_pre_stride + e) : *(const uint4*)(p.u + row * p.u_stride + e), uu);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            y[i] = g[c][i] * __builtin_fmaf((x[c][i] - mean) * rstd, gm[i], bt[i]);
            if (p.u_pre) {
              y[i] = round_bf16(y[i]) * silu_grad(uu[i]);     // (du in bf16, as the attention's dq, dk, dv are)
              uu[i] = round_bf16(silu(uu[i]));
            }
            g[c][i] *= uu[i];
          }
          *(uint4*)(p.du + row * p.du_stride + e) = pack8(y);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float xh = (x[c][i] - mean) * rstd;
          const float gn = g[c][i];
          x[c][i] = xh;
          dg[c][i] = __builtin_fmaf(gn, xh, dg[c][i]);
          db[c][i] += gn;
          const float gx = gn * gm[i];
          g[c][i] = gx;
          s1 += gx;
          s2 = __builtin_fmaf(gx, xh, s2);
        }
      }
    }
    const float c1 = group_sum<LPR>(s1) * inv_w, c2 = group_sum<LPR>(s2) * inv_w;
    bf16_t* dr = p.da + row * p.da_stride;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int e = (c * LPR + lane) * 8;
      if (e < p.width) {
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = rstd * (g[c][i] - c1 - x[c][i] * c2);
        if (p.add) {
          float more[8];
          unpack8(*(const uint4*)(p.add + row * p.add_stride + e), more);
#pragma unroll
          for (int i = 0; i < 8; ++i) y[i] = round_bf16(y[i]) + more[i];      // (each share a bf16 gradient of its own)
        }
        *(uint4*)(dr + e) = pack8(y);
      }
    }
  }
  // the workgroup's column sums: every wave gets here, whatever rows it had
  float* part = p.partial + (int64_t)blockIdx.x * (2 * p.width);
#pragma unroll
  for (int half = 0; half < 2; ++half) {
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float v = half == 0 ? dg[c][i] : db[c][i];
        // (the row groups of a wave hold the same columns)
#pragma unroll
        for (int d = 32; d >= LPR; d >>= 1) v += __shfl_xor(v, d, 64);
        if ((threadIdx.x & 63) < LPR) red[w][(c * LPR + lane) * 8 + i] = v;
      }
    __syncthreads();
    for (int col = threadIdx.x; col < p.width; col += 256)
      part[half * p.width + col] = (red[0][col] + red[1][col]) + (red[2][col] + red[3][col]);
    __syncthreads();
  }
}

// out[col] = sum over the nb partial rows of part[.][col], rows added in a fixed order; columns
// [0, width) go to dgamma, [width, 2 width) to dbeta.  nb = 0 writes zeros.  A workgroup of 1024
// threads takes 32 columns: 32 groups of threads each add every 32nd row (four sums in flight per
// thread: the loop is nothing but dependent loads otherwise), then the groups' sums are added through LDS.
template <typename T>
__global__ __launch_bounds__(1024) void hstu_colsum(const float* __restrict__ part, int nb, int width, T* __restrict__ dgamma,
                                                    T* __restrict__ dbeta) {
  __shared__ float red[32][33];
  const int cl = threadIdx.x & 31, rg = threadIdx.x >> 5;
  const int col = blockIdx.x * 32 + cl, n2 = 2 * width;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
  if (col < n2) {
    const float* pc = part + col;
    int r = rg;
    for (; r + 96 < nb; r += 128) {
      s0 += pc[(int64_t)r * n2];
      s1 += pc[(int64_t)(r + 32) * n2];
      s2 += pc[(int64_t)(r + 64) * n2];
      s3 += pc[(int64_t)(r + 96) * n2];
    }
    for (; r < nb; r += 32) s0 += pc[(int64_t)r * n2];
  }
  red[rg][cl] = (s0 + s1) + (s2 + s3);
  __syncthreads();
  if (rg == 0 && col < n2) {
    float s = 0.f;
#pragma unroll
    for (int g = 0; g < 32; ++g) s += red[g][cl];
    if (col < width) dgamma[col] = (T)s; else dbeta[col - width] = (T)s;
  }
}

// lanes per row of the norm kernels
int lanes_per_row(int width) { return width <= 64 ? 8 : width <= 128 ? 16 : width <= 256 ? 32 : 64; }

// workgroups of the backward kernel for this many rows (each walks over rows with the grid's stride)
int norm_gate_bwd_blocks(int64_t rows, int width) {
  const int64_t per = 4 * (64 / lanes_per_row(width)), nb = (rows + per - 1) / per;
  return (int)(nb < 1 ? 1 : (nb > 1024 ? 1024 : nb));
}

struct EmbedNormParams {
  const int64_t* ids;
  const int64_t* positions;
  const bf16_t* table;
  const bf16_t* pos_table;
  const bf16_t* gamma;
  const bf16_t* beta;
  bf16_t* out;
  const int32_t* row_map;  // token r takes entry row_map[r] of ids (its row in the padded batch), or null: entry r
  int32_t L;               // with positions null: the position is that entry's index modulo L
  int64_t rows, vocab, table_stride, n_positions;
  int32_t width;
  float eps, scale;
  int32_t round_steps;     // the scaled row and the sum are each rounded to bf16, as separate steps would leave them
  bf16_t* sums;            // the rows before the norm, for the gradients; or null
  int64_t* keys;           // the table rows taken, for the gradients; or null
  int32_t* outside;        // raised where an index lies outside its table; or null
  const uint8_t* mask;     // or null: the batch's mask, whose lengths the first `mask_groups` workgroups write
  int32_t* lens;
  int32_t* bad;
  int32_t mask_B, mask_L;
  uint32_t mask_groups;
};

// The length of row b of an end-padded batch's mask (bytes), by one wavefront; *bad is raised by a row that is not a run of non-zero bytes
// followed by zeros.
__device__ __forceinline__ void mask_length(const uint8_t* __restrict__ mask, int b, int L, int lane, int32_t* __restrict__ lens, int32_t* __restrict__ bad) {
  const uint8_t* row = mask + (int64_t)b * L;
  int n = 0, last = -1;
  for (int i = lane; i < L; i += 64) {
    const bool on = row[i] != 0;
    n += on ? 1 : 0;
    last = on ? i : last;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    n += __shfl_xor(n, d, 64);
    const int o = __shfl_xor(last, d, 64);
    last = last > o ? last : o;
  }
  if (lane == 0) {
    lens[b] = n;
    if (last + 1 != n) *bad = 1;
  }
}

// Rows on lanes as in hstu_norm_gate: a token's table row (and position row) is gathered into registers, normalised
// there and written once.  In training the gathered rows and their ids are stored next to it (as many bytes again): the
// backward then works on its own copies, so that neither the ids nor the tables have to stay as they were until it runs.
// With a mask a few more workgroups count its rows: what both do is little beside a launch (32 x 50, width 64: 4.0 + 3.6 us as two).
template <int CH, int LPR>
__global__ __launch_bounds__(256) void hstu_embed_norm(const EmbedNormParams p) {
  constexpr int RPW = 64 / LPR;
  if (blockIdx.x < p.mask_groups) {
    const int b = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (b < p.mask_B) mask_length(p.mask, b, p.mask_L, threadIdx.x & 63, p.lens, p.bad);
    return;
  }
  const int lane = threadIdx.x & (LPR - 1);
  const int64_t row = ((int64_t)(blockIdx.x - p.mask_groups) * 4 + (threadIdx.x >> 6)) * RPW + ((threadIdx.x & 63) / LPR);
  if (row >= p.rows) return;
  const int64_t at = p.row_map ? p.row_map[row] : row;
  int64_t id = p.ids[at];
  if (p.outside) {
    id += id < 0 ? p.vocab : 0;
    if (id < 0 || id >= p.vocab) *p.outside = 1;
  }
  id = id < 0 ? 0 : (id >= p.vocab ? p.vocab - 1 : id);
  if (p.keys && lane == 0) p.keys[row] = id;
  const bf16_t* er = p.table + id * p.table_stride;
  const bf16_t* pr = nullptr;
  if (p.pos_table) {
    int64_t ps = p.positions ? p.positions[row] : at % p.L;
    if (p.outside && (ps < 0 || ps >= p.n_positions)) *p.outside = 1;
    ps = ps < 0 ? 0 : (ps >= p.n_positions ? p.n_positions - 1 : ps);
    pr = p.pos_table + ps * (int64_t)p.width;
  }
  float x[CH][8];
  float sum = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int e = (c * LPR + lane) * 8;
    if (e < p.width) {
      unpack8(*(const uint4*)(er + e), x[c]);
      float pe[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (pr) unpack8(*(const uint4*)(pr + e), pe);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        x[c][i] = p.round_steps ? round_bf16(round_bf16(x[c][i] * p.scale) + pe[i]) : __builtin_fmaf(x[c][i], p.scale, pe[i]);
      if (p.sums) *(uint4*)(p.sums + row * (int64_t)p.width + e) = pack8(x[c]);
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += x[c][i];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[c][i] = 0.f;
    }
  }
  const float mean = group_sum<LPR>(sum) / (float)p.width;
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int e = (c * LPR + lane) * 8;
    if (e < p.width) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float d = x[c][i] - mean;
        ss += d * d;
      }
    }
  }
  const float rstd = __builtin_amdgcn_rsqf(group_sum<LPR>(ss) / (float)p.width + p.eps);
  bf16_t* orow = p.out + row * (int64_t)p.width;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int e = (c * LPR + lane) * 8;
    if (e < p.width) {
      float g[8], b[8], y[8];
      unpack8(*(const uint4*)(p.gamma + e), g);
      unpack8(*(const uint4*)(p.beta + e), b);
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = __builtin_fmaf((x[c][i] - mean) * rstd, g[i], b[i]);
      *(uint4*)(orow + e) = pack8(y);
    }
  }
}

// ---- a batch's packing --------------------------------------------------

// Where the tokens of a padded batch go when it is packed: offsets[b] = the sum of the lengths before b, row_map[t] = the
// padded row b L + i of packed token t, total = the number of tokens.  One workgroup per sequence; each adds up the lengths
// before its own (B of them: at most a few loads per thread).
template <typename T>
__global__ __launch_bounds__(256) void hstu_pack_plan_kernel(const T* __restrict__ lens, int B, int L, int32_t* __restrict__ offsets,
                                                      int32_t* __restrict__ row_map, int32_t* __restrict__ total) {
  __shared__ int part[4];
  const int b = blockIdx.x, tid = threadIdx.x;
  auto len = [&](int x) {
    const int64_t n = (int64_t)lens[x];
    return (int)(n < 0 ? 0 : (n > L ? L : n));
  };
  int sum = 0;
  for (int x = tid; x < b; x += 256) sum += len(x);
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 64);
  if ((tid & 63) == 0) part[tid >> 6] = sum;
  __syncthreads();
  const int off = part[0] + part[1] + part[2] + part[3], n = len(b);
  if (tid == 0) {
    offsets[b] = off;
    if (b == B - 1) {
      offsets[B] = off + n;
      *total = off + n;
    }
  }
  for (int i = tid; i < n; i += 256) row_map[off + i] = b * L + i;
}

// Lengths of an end-padded batch from its mask, one row per wavefront.
__global__ __launch_bounds__(256) void hstu_mask_lengths_kernel(const uint8_t* __restrict__ mask, int B, int L, int32_t* __restrict__ lens,
                                                         int32_t* __restrict__ bad) {
  const int b = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (b < B) mask_length(mask, b, L, lane, lens, bad);
}

// ---- gradients of the embedding tables ----------------------------------

// The gradient of rows gathered from a table: out[v] = the sum of scale * g[t] over the tokens t with key(t) = v, v in [0, V), and
// zeros for the others.  Keys are ids (clamped like the gather) or, with L, positions.  The terms of a key are added in the order
// of the tokens and every partial sum is rounded to bf16 (rows of up to 64 elements: kept in fp32): the arithmetic of torch's
// gather backward, whose kernel did this before (one wavefront per 32 table columns' run of tokens, reading and writing the sum in memory
// for every token: 3.5 ms of a training step of 78 k tokens over 100 k popular and unpopular items, and as much for the positions).
//   A popular key has thousands of tokens and most have none or one.  The tokens are put in order by key (counted, room reserved
// per key, placed: no sort of the whole), a key's run is put in order by token, and the runs are summed in registers: short ones by
// one wavefront each, long ones by one wavefront per 128 columns with 64 rows in flight (the chain of additions is 20 cycles a
// row, the memory latency behind it over a thousand).
constexpr int EG_SHORT = 32;         // tokens of a run that one wavefront orders and sums by itself
constexpr int EG_WINDOW = 1 << 19;   // tokens whose bits fit the LDS of the ordering of a long run
struct EmbedGradParams {
  const bf16_t* g;
  bf16_t* out;
  const int64_t* ids;
  const int64_t* positions;
  const int32_t* row_map;
  int64_t T, V, g_stride, out_stride;
  int32_t L, width, by_position;
  int32_t round_sums;  // every partial sum rounded to bf16
  float scale;
  int32_t* count;      // [V]: tokens of a key, then where its run starts
  int32_t* rank;       // [T]: a token's place in its run
  int32_t* order;      // [T]: tokens by key
  int32_t* heads;      // [4]: tokens placed, short runs, long runs
  int4* shorts;        // {key, first place, tokens, -}
  int4* longs;
  int32_t* sorted;     // [T]: the long runs' tokens in order
};
__device__ __forceinline__ int64_t eg_key(const EmbedGradParams& p, int64_t t) {
  const int64_t at = p.row_map ? p.row_map[t] : t;
  int64_t k = p.by_position ? (p.positions ? p.positions[t] : at % p.L) : p.ids[at];
  return k < 0 ? 0 : (k >= p.V ? p.V - 1 : k);
}
__global__ __launch_bounds__(256) void hstu_eg_clear(const EmbedGradParams p) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < p.V) p.count[i] = 0;
  if (i < 4) p.heads[i] = 0;
}
__global__ __launch_bounds__(256) void hstu_eg_count(const EmbedGradParams p) {
  // one addition per wavefront and key: the tokens of a popular key would otherwise queue at its counter one by one
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const int key = t < p.T ? (int)eg_key(p, t) : -1;
  int leader = lane, rank = 0, members = 0;
  uint64_t left = __builtin_amdgcn_ballot_w64(key >= 0);
  while (left) {
    const int first = __builtin_ctzll(left);
    const uint64_t same = __builtin_amdgcn_ballot_w64(key == __builtin_amdgcn_readlane(key, first));
    if ((same >> lane) & 1) {
      leader = first;
      rank = __builtin_popcountll(same & ((1ull << lane) - 1));
      members = __builtin_popcountll(same);
    }
    left &= ~same;
  }
  int base = 0;
  if (key >= 0 && leader == lane) base = atomicAdd(&p.count[key], members);
  base = __shfl(base, leader, 64);
  if (t < p.T) p.rank[t] = base + rank;
}
// Each workgroup reserves room for its 256 keys with one addition per counter, and clears the rows of those without a token.
__global__ __launch_bounds__(256) void hstu_eg_reserve(const EmbedGradParams p) {
  __shared__ int sums[4][3], base[3];
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int n = v < p.V ? p.count[v] : 0;
  const int mine[3] = {n, n > 0 && n <= EG_SHORT ? 1 : 0, n > EG_SHORT ? 1 : 0};
  int at[3];
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    int s = mine[x];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(s, d, 64);
      s += lane >= d ? o : 0;
    }
    at[x] = s - mine[x];
    if (lane == 63) sums[w][x] = s;
  }
  __syncthreads();
  if (threadIdx.x < 3) base[threadIdx.x] = atomicAdd(&p.heads[threadIdx.x], sums[0][threadIdx.x] + sums[1][threadIdx.x] + sums[2][threadIdx.x] + sums[3][threadIdx.x]);
  __syncthreads();
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    at[x] += base[x];
    for (int y = 0; y < w; ++y) at[x] += sums[y][x];
  }
  if (n > 0) {
    p.count[v] = at[0];
    const int4 run = {(int)v, at[0], n, 0};
    if (n <= EG_SHORT) p.shorts[at[1]] = run; else p.longs[at[2]] = run;
  }
  // the rows of keys without a token, the whole wave one at a time
  uint64_t empty = __builtin_amdgcn_ballot_w64(v < p.V && n == 0);
  const int64_t v0 = v - lane;
  while (empty) {
    const int x = __builtin_ctzll(empty);
    empty &= empty - 1;
    bf16_t* o = p.out + (v0 + x) * p.out_stride;
    for (int e = 8 * lane; e < p.width; e += 512) *(uint4*)(o + e) = uint4{0u, 0u, 0u, 0u};
  }
}
__global__ __launch_bounds__(256) void hstu_eg_place(const EmbedGradParams p) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t < p.T) p.order[p.count[eg_key(p, t)] + p.rank[t]] = (int32_t)t;
}
// One wavefront per short run: its tokens in order by counting the smaller ones, then their rows, four in flight.
__global__ __launch_bounds__(256) void hstu_eg_short(const EmbedGradParams p) {
  __shared__ int tokens[4][EG_SHORT];
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (i >= p.heads[1]) return;
  const int4 run = p.shorts[i];
  const int n = run.z;
  const int mine = lane < n ? p.order[run.y + lane] : 0x7fffffff;
  int r = 0;
  for (int x = 0; x < n; ++x) r += __shfl(mine, x, 64) < mine ? 1 : 0;
  if (lane < n) tokens[w][r] = mine;
  __builtin_amdgcn_wave_barrier();
  for (int e = 8 * lane; e < p.width; e += 512) {
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int x = 0; x < n; x += 4) {
      uint4 v[4];
#pragma unroll
      for (int y = 0; y < 4; ++y) v[y] = *(const uint4*)(p.g + (int64_t)tokens[w][x + y < n ? x + y : x] * p.g_stride + e);
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        if (x + y < n) {
          float f[8];
          unpack8(v[y], f);
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            s[k] += p.scale == 1.f ? f[k] : round_bf16(f[k] * p.scale);
            s[k] = p.round_sums ? round_bf16(s[k]) : s[k];
          }
        }
      }
    }
    *(uint4*)(p.out + (int64_t)run.x * p.out_stride + e) = pack8(s);
  }
}
// One workgroup per long run: its tokens' bits set in LDS, read back in order.
__global__ __launch_bounds__(256) void hstu_eg_order(const EmbedGradParams p) {
  extern __shared__ __attribute__((aligned(16))) uint32_t bits[];
  __shared__ int sums[4];
  if ((int)blockIdx.x >= p.heads[2]) return;
  const int4 run = p.longs[blockIdx.x];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  int done = 0;
  for (int64_t t0 = 0; t0 < p.T; t0 += EG_WINDOW) {
    const int span = (int)(p.T - t0 < EG_WINDOW ? p.T - t0 : EG_WINDOW), words = (span + 31) >> 5;
    for (int x = tid; x < words; x += 256) bits[x] = 0u;
    __syncthreads();
    for (int x = tid; x < run.z; x += 256) {
      const int64_t t = p.order[run.y + x] - t0;
      if (t >= 0 && t < span) atomicOr(&bits[t >> 5], 1u << (t & 31));
    }
    __syncthreads();
    // every thread a stretch of words: count, prefix sum, write
    const int per = (words + 255) / 256, x0 = tid * per < words ? tid * per : words, x1 = x0 + per < words ? x0 + per : words;
    int c = 0;
    for (int x = x0; x < x1; ++x) c += __builtin_popcount(bits[x]);
    int s = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(s, d, 64);
      s += lane >= d ? o : 0;
    }
    if (lane == 63) sums[w] = s;
    __syncthreads();
    int at = done + s - c;
    for (int y = 0; y < w; ++y) at += sums[y];
    for (int x = x0; x < x1; ++x) {
      uint32_t m = bits[x];
      while (m) {
        p.sorted[run.y + at++] = (int32_t)(t0 + 32 * x + __builtin_ctz(m));
        m &= m - 1;
      }
    }
    done += sums[0] + sums[1] + sums[2] + sums[3];
    __syncthreads();
  }
}
// One wavefront per long run and 128 columns, two columns per lane.  Its rows come 64 at a time, four to an instruction (16 lanes to the
// 256 bytes of one), two or three such batches under way.  Loads of one row each held 64 rows at most -- the counter of outstanding loads
// goes to 63 -- and waited for memory, 115 clocks a row; here the additions bound it, 60.  (78 k rows of 512, the most popular key
// 4700 of them: 225 -> 119 us.)
// WIDE: partial sums rounded to bf16.
template <bool WIDE, bool SCALED>
__global__ __launch_bounds__(64) void hstu_eg_long(const EmbedGradParams p) {
  if ((int)blockIdx.x >= p.heads[2]) return;
  const int4 run = p.longs[blockIdx.x];
  const int lane = threadIdx.x, grp = lane >> 4;
  const int32_t* tok = p.sorted + run.y;
  const int e = blockIdx.y * 128 + 8 * (lane & 15);      // of the 16 bytes a lane loads; it sums columns e + 2 grp and the next
  const bool on = e < p.width;
  const bf16_t* g = p.g + (on ? e : 0);
  float s0 = 0.f, s1 = 0.f;
  constexpr int BATCH = 64, LOADS = BATCH / 4;
  uint4 a[LOADS], b[LOADS], c[LOADS];
  // A lane holds one of 64 tokens.  Tokens are asked for ahead of the rows that are under way when they are needed: loads return in
  // order, so that waiting for tokens behind rows would empty the pipeline at every batch.
  auto tokens = [&](int x) __attribute__((always_inline)) { return tok[x + lane < run.z ? x + lane : 0]; };
  auto fetch = [&](uint4 (&v)[LOADS], int held) __attribute__((always_inline)) {
#pragma unroll
    for (int y = 0; y < LOADS; ++y) v[y] = *(const uint4*)(g + (int64_t)__shfl(held, 4 * y + grp, 64) * p.g_stride);
    __builtin_amdgcn_sched_barrier(0);
  };
  // (a value rounded to bf16 as the upper half of a word is that value in fp32: one conversion, no shift behind it)
  auto rounded = [](float x) __attribute__((always_inline)) { return __builtin_bit_cast(float, pack2(0.f, x)); };
  auto add = [&](const uint4 (&v)[LOADS], int n, auto whole_) __attribute__((always_inline)) {
    constexpr bool whole = decltype(whole_)::value;
#pragma unroll
    for (int y = 0; y < LOADS; ++y) {
      // lanes of row grp with words 0 .. 3 to rows 0 .. 3 with the lanes' word grp
      const auto x0 = __builtin_amdgcn_permlane32_swap(v[y].x, v[y].z, false, false), x1 = __builtin_amdgcn_permlane32_swap(v[y].y, v[y].w, false, false);
      const uint32_t r00 = x0[0], r01 = x0[1], r10 = x1[0], r11 = x1[1];
      const auto y0 = __builtin_amdgcn_permlane16_swap(r00, r10, false, false), y1 = __builtin_amdgcn_permlane16_swap(r01, r11, false, false);
      const uint32_t row[4] = {y0[0], y0[1], y1[0], y1[1]};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t u = whole || 4 * y + j < n ? row[j] : 0u;      // past the run's end: zeros
        float f0 = __builtin_bit_cast(float, u << 16), f1 = __builtin_bit_cast(float, u & 0xffff0000u);
        if (SCALED) { f0 = rounded(f0 * p.scale); f1 = rounded(f1 * p.scale); }
        s0 += f0;
        s1 += f1;
        if (WIDE) { s0 = rounded(s0); s1 = rounded(s1); }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int t0 = tokens(0), t1 = tokens(BATCH), t2 = tokens(2 * BATCH), t3 = tokens(3 * BATCH);
  fetch(a, t0);
  fetch(b, t1);
  for (int x = 0;;) {
    // batch m at x: the tokens of m + 4, the rows of m + 2, the sum of m
    auto step = [&](const uint4 (&sum)[LOADS], uint4 (&load)[LOADS]) __attribute__((always_inline)) {
      const int t4 = tokens(x + 4 * BATCH);
      __builtin_amdgcn_sched_barrier(0);
      fetch(load, t2);
      if (run.z - x >= BATCH) add(sum, BATCH, std::true_type{});
      else add(sum, run.z - x, std::false_type{});
      t2 = t3;
      t3 = t4;
      x += BATCH;
    };
    step(a, c);
    if (x >= run.z) break;
    step(b, a);
    if (x >= run.z) break;
    step(c, b);
    if (x >= run.z) break;
  }
  if (on) *(uint32_t*)(p.out + (int64_t)run.x * p.out_stride + e + 2 * grp) = pack2(s0, s1);
}

void launch_norm_bwd(const NormGateBwdParams& p, int nb, hipStream_t st) {
  const dim3 grid((unsigned)nb), block(256);
  const int lpr = lanes_per_row(p.width), ch = (p.width + 511) / 512;
  if (lpr == 8) hipLaunchKernelGGL((hstu_norm_gate_bwd<1, 8>), grid, block, 0, st, p);
  else if (lpr == 16) hipLaunchKernelGGL((hstu_norm_gate_bwd<1, 16>), grid, block, 0, st, p);
  else if (lpr == 32) hipLaunchKernelGGL((hstu_norm_gate_bwd<1, 32>), grid, block, 0, st, p);
  else if (ch <= 1) hipLaunchKernelGGL((hstu_norm_gate_bwd<1, 64>), grid, block, 0, st, p);
  else if (ch <= 2) hipLaunchKernelGGL((hstu_norm_gate_bwd<2, 64>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((hstu_norm_gate_bwd<4, 64>), grid, block, 0, st, p);
}

struct EmbedGradPlan {
  int64_t shorts, longs;         // most there can be
  size_t count, rank, order, heads, short_list, long_list, sorted, total;
};
EmbedGradPlan embed_grad_plan(int64_t T, int64_t V) {
  EmbedGradPlan w;
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  w.longs = T / (EG_SHORT + 1) < V ? T / (EG_SHORT + 1) : V;
  w.shorts = T < V ? T : V;
  size_t at = 0;
  w.count = at; at += up((size_t)V * 4);
  w.rank = at; at += up((size_t)T * 4);
  w.order = at; at += up((size_t)T * 4);
  w.heads = at; at += 256;
  w.short_list = at; at += up((size_t)w.shorts * 16);
  w.long_list = at; at += up((size_t)w.longs * 16);
  w.sorted = at; at += up((size_t)T * 4);
  w.total = at;
  return w;
}

// ---- SiLU's gradient in place: d *= silu'(pre), rows of `width` elements with strides
__global__ __launch_bounds__(256) void hstu_silu_bwd_kernel(bf16_t* d, const bf16_t* pre, int64_t rows, int width, int64_t d_stride, int64_t pre_stride) {
  const int pieces = width / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = i / pieces;
  if (row >= rows) return;
  const int e = (int)(i - row * pieces) * 8;
  float x[8], z[8];
  unpack8(*(const uint4*)(d + row * d_stride + e), x);
  unpack8(*(const uint4*)(pre + row * pre_stride + e), z);
#pragma unroll
  for (int k = 0; k < 8; ++k) x[k] *= silu_grad(z[k]);
  *(uint4*)(d + row * d_stride + e) = pack8(x);
}

}  // namespace

extern "C" {

int hstu_block_abi_version(void) { return HSTU_BLOCK_ABI_VERSION; }

const char* hstu_block_last_error(void) { return g_err; }

int hstu_norm_gate_fwd(const HstuNormGateArgs* a, void* stream) {
  HstuNormGateArgs own;
  a = block_today(a, own, offsetof(HstuNormGateArgs, seq_offsets), sizeof(HstuNormGateArgs));
  if (!a) return block_fail(HSTU_BLOCK_ERR_NULL, "args is null");
  if (a->struct_size != sizeof(HstuNormGateArgs) || a->version != HSTU_BLOCK_ABI_VERSION)
    return block_fail(HSTU_BLOCK_ERR_VERSION, "norm-gate args struct_size/version (%u/%u) do not match this library (%zu/%d)",
                a->struct_size, a->version, sizeof(HstuNormGateArgs), HSTU_BLOCK_ABI_VERSION);
  if (a->rows < 0 || a->width < 8 || a->width > 8192 || (a->width & 7))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "rows >= 0 and width a multiple of 8 in [8, 8192] expected, got rows=%lld width=%d",
                (long long)a->rows, a->width);
  g_err[0] = 0;
  if (a->rows == 0) return HSTU_BLOCK_OK;
  if (!a->a || !a->out || !a->gamma || !a->beta) return block_fail(HSTU_BLOCK_ERR_NULL, "a, out, gamma and beta must be non-null");
  if (!block_aligned16(a->a) || !block_aligned16(a->u) || !block_aligned16(a->out) || !block_aligned16(a->gamma) || !block_aligned16(a->beta) ||
      (a->a_stride & 7) || (a->out_stride & 7) || a->a_stride < a->width || a->out_stride < a->width ||
      (a->u && ((a->u_stride & 7) || a->u_stride < a->width)))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "pointers must be 16-byte aligned, row strides multiples of 8 elements and >= width");
  if ((a->rows + 3) / 4 > 0x7fffffffLL) return block_fail(HSTU_BLOCK_ERR_SHAPE, "too many rows");
  if (a->seq_offsets && (a->u || a->L < 1)) return block_fail(HSTU_BLOCK_ERR_SHAPE, "a padded output takes L >= 1 and no gate");
  NormGateParams p;
  p.a = (const bf16_t*)a->a; p.u = (const bf16_t*)a->u; p.out = (bf16_t*)a->out;
  p.gamma = (const bf16_t*)a->gamma; p.beta = (const bf16_t*)a->beta;
  p.rows = a->rows; p.a_stride = a->a_stride; p.u_stride = a->u_stride; p.out_stride = a->out_stride;
  p.width = a->width; p.eps = a->eps;
  p.seq_offsets = a->seq_offsets; p.L = a->L;
  hipStream_t st = (hipStream_t)stream;
  const int lpr = lanes_per_row(a->width), per = 4 * (64 / lpr), ch = (a->width + 511) / 512;
  const dim3 grid((unsigned)((a->rows + per - 1) / per)), block(256);
  if (lpr == 8) hipLaunchKernelGGL((hstu_norm_gate<1, 8>), grid, block, 0, st, p);
  else if (lpr == 16) hipLaunchKernelGGL((hstu_norm_gate<1, 16>), grid, block, 0, st, p);
  else if (lpr == 32) hipLaunchKernelGGL((hstu_norm_gate<1, 32>), grid, block, 0, st, p);
  else if (ch <= 1) hipLaunchKernelGGL((hstu_norm_gate<1, 64>), grid, block, 0, st, p);
  else if (ch <= 2) hipLaunchKernelGGL((hstu_norm_gate<2, 64>), grid, block, 0, st, p);
  else if (ch <= 4) hipLaunchKernelGGL((hstu_norm_gate<4, 64>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((hstu_norm_gate<16, 64>), grid, block, 0, st, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "norm-gate kernel launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

size_t hstu_norm_gate_bwd_workspace_bytes(int64_t rows, int32_t width) {
  if (rows < 0 || width < 8) return 0;
  return (size_t)norm_gate_bwd_blocks(rows, width) * 2u * (size_t)width * sizeof(float);
}

}  // extern "C"

template <typename T>
static int norm_gate_bwd(const HstuNormGateBwdArgs* a, void* stream) {
  HstuNormGateBwdArgs own;
  a = block_today(a, own, offsetof(HstuNormGateBwdArgs, u_pre), sizeof(HstuNormGateBwdArgs));
  if (!a) return block_fail(HSTU_BLOCK_ERR_NULL, "args is null");
  if (a->struct_size != sizeof(HstuNormGateBwdArgs) || a->version != HSTU_BLOCK_ABI_VERSION)
    return block_fail(HSTU_BLOCK_ERR_VERSION, "norm-gate backward args struct_size/version (%u/%u) do not match this library (%zu/%d)",
                a->struct_size, a->version, sizeof(HstuNormGateBwdArgs), HSTU_BLOCK_ABI_VERSION);
  if (a->rows < 0 || a->width < 8 || a->width > 2048 || (a->width & 7))
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "rows >= 0 and width a multiple of 8 in [8, 2048] expected, got rows=%lld width=%d",
                (long long)a->rows, a->width);
  g_err[0] = 0;
  if (!a->dgamma || !a->dbeta) return block_fail(HSTU_BLOCK_ERR_NULL, "dgamma and dbeta must be non-null");
  hipStream_t st = (hipStream_t)stream;
  const int nb = a->rows == 0 ? 0 : norm_gate_bwd_blocks(a->rows, a->width);
  if (nb > 0) {
    if (!a->a || !a->dout || !a->da || !a->gamma || !a->beta) return block_fail(HSTU_BLOCK_ERR_NULL, "a, dout, da, gamma and beta must be non-null");
    if ((a->u == nullptr) != (a->du == nullptr)) return block_fail(HSTU_BLOCK_ERR_NULL, "u and du go together (both null: the plain layer norm)");
    if (!block_aligned16(a->a) || !block_aligned16(a->u) || !block_aligned16(a->dout) || !block_aligned16(a->da) || !block_aligned16(a->du) ||
        !block_aligned16(a->gamma) || !block_aligned16(a->beta) ||
        (a->a_stride & 7) || (a->dout_stride & 7) || (a->da_stride & 7) ||
        a->a_stride < a->width || a->dout_stride < a->width || a->da_stride < a->width ||
        (a->u && ((a->u_stride & 7) || (a->du_stride & 7) || a->u_stride < a->width || a->du_stride < a->width)))
      return block_fail(HSTU_BLOCK_ERR_SHAPE, "pointers must be 16-byte aligned, row strides multiples of 8 elements and >= width");
    const size_t need = hstu_norm_gate_bwd_workspace_bytes(a->rows, a->width);
    if (!a->workspace || a->workspace_bytes < need || ((uintptr_t)a->workspace & 3u))
      return block_fail(HSTU_BLOCK_ERR_WORKSPACE, "workspace of %zu bytes needed (hstu_norm_gate_bwd_workspace_bytes), got %zu", need,
                  a->workspace ? a->workspace_bytes : (size_t)0);
    if ((a->u_pre && (!a->u || !block_aligned16(a->u_pre) || (a->u_pre_stride & 7) || a->u_pre_stride < a->width)) ||
        (a->add && (!block_aligned16(a->add) || (a->add_stride & 7) || a->add_stride < a->width)))
      return block_fail(HSTU_BLOCK_ERR_SHAPE, "u_pre (with a gate) and add: 16-byte aligned, row strides multiples of 8 elements and >= width");
    NormGateBwdParams p = {};
    p.u_pre = (const bf16_t*)a->u_pre; p.u_pre_stride = a->u_pre_stride;
    p.add = (const bf16_t*)a->add; p.add_stride = a->add_stride; p.row_map = a->row_map;
    p.a = (const bf16_t*)a->a; p.u = (const bf16_t*)a->u; p.dout = (const bf16_t*)a->dout;
    p.gamma = (const bf16_t*)a->gamma; p.beta = (const bf16_t*)a->beta;
    p.da = (bf16_t*)a->da; p.du = (bf16_t*)a->du; p.partial = (float*)a->workspace;
    p.rows = a->rows; p.a_stride = a->a_stride; p.u_stride = a->u_stride; p.dout_stride = a->dout_stride;
    p.da_stride = a->da_stride; p.du_stride = a->du_stride; p.width = a->width; p.eps = a->eps;
    launch_norm_bwd(p, nb, st);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "norm-gate backward kernel launch: %s", hipGetErrorString(e));
  }
  hipLaunchKernelGGL(hstu_colsum<T>, dim3((unsigned)((2 * a->width + 31) / 32)), dim3(1024), 0, st, (const float*)a->workspace, nb, a->width,
                     (T*)a->dgamma, (T*)a->dbeta);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "column-sum kernel launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

extern "C" {

int hstu_norm_gate_bwd(const HstuNormGateBwdArgs* a, void* stream) { return norm_gate_bwd<float>(a, stream); }

// (a launch for each vector's conversion otherwise: 4 us each, twenty of them in a ranking model's step)
int hstu_norm_gate_bwd_rounded(const HstuNormGateBwdArgs* a, void* stream) { return norm_gate_bwd<bf16_t>(a, stream); }

int hstu_embed_norm_fwd(const HstuEmbedNormArgs* a, void* stream) { return hstu_embed_norm_mask_fwd(a, nullptr, 0, 0, nullptr, nullptr, stream); }

int hstu_embed_norm_mask_fwd(const HstuEmbedNormArgs* a, const uint8_t* mask, int32_t mask_B, int32_t mask_L, int32_t* lens, int32_t* bad, void* stream) {
  HstuEmbedNormArgs own;
  a = block_today(a, own, offsetof(HstuEmbedNormArgs, row_map), offsetof(HstuEmbedNormArgs, sums));
  if (!a) return block_fail(HSTU_BLOCK_ERR_NULL, "args is null");
  if (a->struct_size != sizeof(HstuEmbedNormArgs) || a->version != HSTU_BLOCK_ABI_VERSION)
    return block_fail(HSTU_BLOCK_ERR_VERSION, "embed-norm args struct_size/version (%u/%u) do not match this library (%zu/%d)",
                a->struct_size, a->version, sizeof(HstuEmbedNormArgs), HSTU_BLOCK_ABI_VERSION);
  if (a->rows < 0 || a->width < 8 || a->width > 8192 || (a->width & 7) || a->vocab < 1)
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "rows >= 0, vocab >= 1 and width a multiple of 8 in [8, 8192] expected, got rows=%lld vocab=%lld width=%d",
                (long long)a->rows, (long long)a->vocab, a->width);
  g_err[0] = 0;
  if (mask && (!lens || !bad)) return block_fail(HSTU_BLOCK_ERR_NULL, "lens and bad must be non-null");
  if (mask && (mask_B < 1 || mask_L < 1)) return block_fail(HSTU_BLOCK_ERR_SHAPE, "bad batch B=%d L=%d", mask_B, mask_L);
  if (a->rows == 0) return mask ? hstu_mask_lengths(mask, mask_B, mask_L, lens, bad, stream) : HSTU_BLOCK_OK;
  if (!a->ids || !a->table || !a->out || !a->gamma || !a->beta) return block_fail(HSTU_BLOCK_ERR_NULL, "ids, table, out, gamma and beta must be non-null");
  if ((a->pos_table != nullptr) != (a->positions != nullptr || a->L > 0) || (a->pos_table && a->n_positions < 1) || a->L < 0)
    return block_fail(HSTU_BLOCK_ERR_NULL, "pos_table and positions (or L) go together (with n_positions >= 1)");
  if (!block_aligned16(a->table) || !block_aligned16(a->pos_table) || !block_aligned16(a->out) || !block_aligned16(a->gamma) || !block_aligned16(a->beta) ||
      (a->table_stride & 7) || a->table_stride < a->width)
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "pointers must be 16-byte aligned, table_stride a multiple of 8 elements and >= width");
  if (a->sums && (!a->round_steps || !block_aligned16(a->sums))) return block_fail(HSTU_BLOCK_ERR_SHAPE, "sums go with round_steps and are 16-byte aligned");
  const uint32_t mask_groups = mask ? (uint32_t)((mask_B + 3) / 4) : 0u;
  if ((a->rows + 3) / 4 + (int64_t)mask_groups > 0x7fffffffLL) return block_fail(HSTU_BLOCK_ERR_SHAPE, "too many rows");
  EmbedNormParams p;
  p.ids = a->ids; p.positions = a->positions;
  p.table = (const bf16_t*)a->table; p.pos_table = (const bf16_t*)a->pos_table;
  p.gamma = (const bf16_t*)a->gamma; p.beta = (const bf16_t*)a->beta; p.out = (bf16_t*)a->out;
  p.rows = a->rows; p.vocab = a->vocab; p.table_stride = a->table_stride; p.n_positions = a->n_positions;
  p.width = a->width; p.eps = a->eps; p.scale = a->scale;
  p.row_map = a->row_map; p.L = a->L; p.round_steps = a->round_steps;
  p.sums = (bf16_t*)a->sums; p.keys = a->keys; p.outside = a->outside;
  p.mask = mask; p.lens = lens; p.bad = bad; p.mask_B = mask_B; p.mask_L = mask_L; p.mask_groups = mask_groups;
  hipStream_t st = (hipStream_t)stream;
  const int lpr = lanes_per_row(a->width), per = 4 * (64 / lpr), ch = (a->width + 511) / 512;
  const dim3 grid((unsigned)((a->rows + per - 1) / per) + mask_groups), block(256);
  if (lpr == 8) hipLaunchKernelGGL((hstu_embed_norm<1, 8>), grid, block, 0, st, p);
  else if (lpr == 16) hipLaunchKernelGGL((hstu_embed_norm<1, 16>), grid, block, 0, st, p);
  else if (lpr == 32) hipLaunchKernelGGL((hstu_embed_norm<1, 32>), grid, block, 0, st, p);
  else if (ch <= 1) hipLaunchKernelGGL((hstu_embed_norm<1, 64>), grid, block, 0, st, p);
  else if (ch <= 2) hipLaunchKernelGGL((hstu_embed_norm<2, 64>), grid, block, 0, st, p);
  else if (ch <= 4) hipLaunchKernelGGL((hstu_embed_norm<4, 64>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((hstu_embed_norm<16, 64>), grid, block, 0, st, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "embed-norm kernel launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

size_t hstu_embed_grad_workspace_bytes(int64_t rows, int64_t keys, int32_t width) {
  return rows < 0 || keys < 1 || width < 8 ? 0 : embed_grad_plan(rows, keys).total;
}

int hstu_embed_grad(const HstuEmbedGradArgs* a, void* stream) {
  HstuEmbedGradArgs own;
  a = block_today(a, own, 0, sizeof(HstuEmbedGradArgs));
  if (!a) return block_fail(HSTU_BLOCK_ERR_NULL, "args is null");
  if (a->struct_size != sizeof(HstuEmbedGradArgs) || a->version != HSTU_BLOCK_ABI_VERSION)
    return block_fail(HSTU_BLOCK_ERR_VERSION, "embedding gradient args do not match this library");
  if (a->rows < 0 || a->rows > 0x7fffffff || a->keys < 1 || a->keys > 0x7fffffff || a->width < 8 || (a->width & 7) || a->L < 0)
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "rows >= 0, keys >= 1 and width a multiple of 8 expected");
  if (!a->out || !block_aligned16(a->out) || (a->rows && (!a->g || !block_aligned16(a->g))) || (a->g_stride & 7) || a->g_stride < a->width)
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "g and out must be 16-byte aligned, g_stride a multiple of 8 elements and >= width");
  if (a->rows && !(a->by_position ? (a->positions || a->L > 0) : a->ids != nullptr)) return block_fail(HSTU_BLOCK_ERR_NULL, "the keys are missing");
  const EmbedGradPlan w = embed_grad_plan(a->rows, a->keys);
  if (!a->workspace || a->workspace_bytes < w.total || ((uintptr_t)a->workspace & 255u))
    return block_fail(HSTU_BLOCK_ERR_WORKSPACE, "workspace of %zu bytes needed (hstu_embed_grad_workspace_bytes), 256-byte aligned", w.total);
  char* base = (char*)a->workspace;
  EmbedGradParams p = {};
  p.g = (const bf16_t*)a->g; p.out = (bf16_t*)a->out; p.ids = a->ids; p.positions = a->positions; p.row_map = a->row_map;
  p.T = a->rows; p.V = a->keys; p.g_stride = a->g_stride; p.out_stride = a->width; p.L = a->L; p.width = a->width; p.by_position = a->by_position;
  p.scale = a->scale;
  // (a position's rows in a padded batch were not gathered but broadcast: that gradient is one fp32 sum, rounded once)
  p.round_sums = a->width > 64 && a->by_position != 2;
  p.count = (int32_t*)(base + w.count); p.rank = (int32_t*)(base + w.rank); p.order = (int32_t*)(base + w.order); p.heads = (int32_t*)(base + w.heads);
  p.shorts = (int4*)(base + w.short_list); p.longs = (int4*)(base + w.long_list); p.sorted = (int32_t*)(base + w.sorted);
  hipStream_t st = (hipStream_t)stream;
  const unsigned bv = (unsigned)((p.V + 255) / 256), bt = (unsigned)((p.T + 255) / 256);
  hipLaunchKernelGGL(hstu_eg_clear, dim3(bv), dim3(256), 0, st, p);
  if (bt) hipLaunchKernelGGL(hstu_eg_count, dim3(bt), dim3(256), 0, st, p);
  hipLaunchKernelGGL(hstu_eg_reserve, dim3(bv), dim3(256), 0, st, p);
  if (bt) {
    hipLaunchKernelGGL(hstu_eg_place, dim3(bt), dim3(256), 0, st, p);
    if (w.longs) {
      // (the long runs first: the longest of them is the last to end)
      const int64_t span = p.T < EG_WINDOW ? p.T : EG_WINDOW;
      const int lds = (int)((span + 31) / 32 * 4);
      static int granted[64];
      if (int rc = block_allow_lds((const void*)hstu_eg_order, EG_WINDOW / 8, granted)) return rc;
      hipLaunchKernelGGL(hstu_eg_order, dim3((unsigned)w.longs), dim3(256), lds, st, p);
      const dim3 grid((unsigned)w.longs, (unsigned)((p.width + 127) / 128));
      const bool wide = p.round_sums != 0, scaled = p.scale != 1.f;
      if (wide && scaled) hipLaunchKernelGGL((hstu_eg_long<true, true>), grid, dim3(64), 0, st, p);
      else if (wide) hipLaunchKernelGGL((hstu_eg_long<true, false>), grid, dim3(64), 0, st, p);
      else if (scaled) hipLaunchKernelGGL((hstu_eg_long<false, true>), grid, dim3(64), 0, st, p);
      else hipLaunchKernelGGL((hstu_eg_long<false, false>), grid, dim3(64), 0, st, p);
    }
    hipLaunchKernelGGL(hstu_eg_short, dim3((unsigned)((w.shorts + 3) / 4)), dim3(256), 0, st, p);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "embedding gradient launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

int hstu_pack_plan(const void* lens, int32_t lens_are_64bit, int32_t B, int32_t L, int32_t* seq_offsets, int32_t* row_map, int32_t* total, void* stream) {
  if (!lens || !seq_offsets || !row_map || !total) return block_fail(HSTU_BLOCK_ERR_NULL, "lens, seq_offsets, row_map and total must be non-null");
  if (B < 1 || L < 1 || (int64_t)B * L > 0x7fffffffLL) return block_fail(HSTU_BLOCK_ERR_SHAPE, "bad batch B=%d L=%d", B, L);
  hipStream_t st = (hipStream_t)stream;
  if (lens_are_64bit) hipLaunchKernelGGL(hstu_pack_plan_kernel<int64_t>, dim3((unsigned)B), dim3(256), 0, st, (const int64_t*)lens, B, L, seq_offsets, row_map, total);
  else hipLaunchKernelGGL(hstu_pack_plan_kernel<int32_t>, dim3((unsigned)B), dim3(256), 0, st, (const int32_t*)lens, B, L, seq_offsets, row_map, total);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "pack plan launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

int hstu_mask_lengths(const uint8_t* mask, int32_t B, int32_t L, int32_t* lens, int32_t* bad, void* stream) {
  if (!mask || !lens || !bad) return block_fail(HSTU_BLOCK_ERR_NULL, "mask, lens and bad must be non-null");
  if (B < 1 || L < 1) return block_fail(HSTU_BLOCK_ERR_SHAPE, "bad batch B=%d L=%d", B, L);
  hipLaunchKernelGGL(hstu_mask_lengths_kernel, dim3((unsigned)((B + 3) / 4)), dim3(256), 0, (hipStream_t)stream, mask, B, L, lens, bad);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "mask lengths launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

int hstu_silu_bwd(void* d, int64_t d_stride, const void* pre, int64_t pre_stride, int64_t rows, int32_t width, void* stream) {
  if (rows < 0 || width < 8 || (width & 7) || (d_stride & 7) || (pre_stride & 7) || d_stride < width || pre_stride < width)
    return block_fail(HSTU_BLOCK_ERR_SHAPE, "rows >= 0, width and row strides multiples of 8 expected");
  if (rows == 0) return HSTU_BLOCK_OK;
  if (!d || !pre || !block_aligned16(d) || !block_aligned16(pre)) return block_fail(HSTU_BLOCK_ERR_NULL, "d and pre must be 16-byte aligned");
  const int64_t n = rows * (width / 8);
  hipLaunchKernelGGL(hstu_silu_bwd_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, (bf16_t*)d, (const bf16_t*)pre, rows, width,
                     d_stride, pre_stride);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return block_fail(HSTU_BLOCK_ERR_LAUNCH, "silu backward launch: %s", hipGetErrorString(e));
  return HSTU_BLOCK_OK;
}

}  // extern "C"
