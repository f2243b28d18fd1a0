/* C ABI of libhstu_block.so: the fused steps of the HSTU block that sit on
 * either side of the attention kernel (recml/layers/keras/hstu.py:444-474) and
 * of the model's front end (hstu.py:593-601), for gfx950.  bf16 tensors, row-major, on the current device; fp32 arithmetic
 * inside.  Plain pointers and sizes: no framework types.
 *
 *   hstu_gemm_silu_fwd    out = silu(x W + bias): the U, Q, K, V projections of
 *                         the normalised input with their activation
 *                         (hstu.py:444-449, the EinsumDense layers of :281-330
 *                         with activation="silu"), as ONE matrix product with
 *                         the activation in its epilogue instead of a pass of
 *                         its own (hstu_gemm's kernels).
 *   hstu_norm_gate_fwd    out = u * layer_norm(attn): the layer norm over
 *                         (heads, head_dim) of the attention output and the U
 *                         gate (hstu.py:471-472) in one pass over memory.
 *   hstu_norm_gate_bwd    the gradients of that step for training: of the
 *                         attention output, of U, of the norm's scale and
 *                         offset (what the framework's autodiff derives from
 *                         hstu.py:471-472); without a gate, the gradients of a
 *                         plain layer norm (the block's input norm,
 *                         hstu.py:442, and the model's final_norm).
 *   hstu_embed_norm_fwd   out = layer_norm(scale * table[ids] + pos_table[positions]):
 *                         the model's front end (hstu.py:593-601: item
 *                         embedding, optional sqrt(D) scale, position
 *                         embedding, final_norm) as one gather pass.
 *
 * Every function returns 0 or a negative HstuBlockStatus; the message of the
 * last failure on the calling thread is at hstu_block_last_error().
 */
#ifndef HSTU_BLOCK_H_
#define HSTU_BLOCK_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Versions since 3 added members at the end of HstuNormGateArgs, HstuNormGateBwdArgs and HstuEmbedNormArgs (4: seq_offsets and L;
 * u_pre, add and row_map; row_map, L and round_steps; 5: sums, keys and outside) and functions; 5 took hstu_embed_norm_bwd away.
 * Callers built against 3 or 4 are taken as they are: their structs say so in struct_size and version, and what they do not have
 * is zero.  Any other pair that does not match is refused (HSTU_BLOCK_ERR_VERSION). */
#define HSTU_BLOCK_ABI_VERSION 5

typedef enum HstuBlockStatus {
  HSTU_BLOCK_OK = 0,
  HSTU_BLOCK_ERR_NULL = -1,
  HSTU_BLOCK_ERR_VERSION = -2,
  HSTU_BLOCK_ERR_SHAPE = -4,
  HSTU_BLOCK_ERR_WORKSPACE = -5,
  HSTU_BLOCK_ERR_LAUNCH = -6,
  HSTU_BLOCK_ERR_BLAS = -7      /* no longer returned (the products were a library's once) */
} HstuBlockStatus;

/* out[t, :] = u[t, :] * (gamma * (a[t, :] - mean_t) * rstd_t + beta), mean and
 * (biased) variance of a[t, :] over its `width` entries, rstd = 1/sqrt(var + eps)
 * (keras LayerNormalization over the last two axes of [.., H, hd] flattened,
 * hstu.py:340-346 and :471-472).  a, u, out: bf16 [rows, width] with the given
 * row strides in elements (u is usually a slice of the fused projection);
 * gamma, beta: bf16 [width].  width a multiple of 8 up to 8192; pointers and
 * row strides multiples of 8 elements (16 bytes).  u may be null: then
 * out = layer_norm(a), the plain norm (u_stride is ignored). */
typedef struct HstuNormGateArgs {
  uint32_t struct_size;   /* sizeof(HstuNormGateArgs)  */
  uint32_t version;       /* HSTU_BLOCK_ABI_VERSION    */
  int64_t rows;
  int32_t width;
  float eps;
  const void* a;
  const void* u;
  void* out;
  int64_t a_stride, u_stride, out_stride;
  const void* gamma;
  const void* beta;
  const int32_t* seq_offsets; /* or null.  Given: out is a padded batch [rows / L][L], sequence b's rows are those of `a` */
  int32_t L, reserved0;       /* from row seq_offsets[b] on, rows past its end (seq_offsets[b + 1]) are zeros; no gate then */
} HstuNormGateArgs;

int hstu_norm_gate_fwd(const HstuNormGateArgs* args, void* stream);

/* Gradients of hstu_norm_gate_fwd for the gradient `dout` of its result (the
 * reference leaves these to autodiff of hstu.py:471-472 and of keras
 * LayerNormalization):
 *   da     bf16 [rows, width]  gradient of a
 *   du     bf16 [rows, width]  gradient of u (usually a slice of the gradient
 *                              of the fused projection: du_stride)
 *   dgamma, dbeta  fp32 [width], overwritten: sums over the rows, added in a
 *                              fixed order (the same bits on every run)
 * a, u, gamma, beta, eps as in the forward call; u and du null together: the
 * gradients of a plain layer norm.  width a multiple of 8 up to 2048; pointers
 * and row strides multiples of 8 elements.  `workspace`: device memory of
 * hstu_norm_gate_bwd_workspace_bytes(rows, width) bytes (one partial row of
 * column sums per workgroup), owned by the caller; the library allocates
 * nothing.  rows = 0 writes zeros to dgamma and dbeta. */
typedef struct HstuNormGateBwdArgs {
  uint32_t struct_size;   /* sizeof(HstuNormGateBwdArgs) */
  uint32_t version;       /* HSTU_BLOCK_ABI_VERSION      */
  int64_t rows;
  int32_t width;
  float eps;
  const void* a;
  const void* u;
  const void* dout;
  void* da;
  void* du;
  int64_t a_stride, u_stride, dout_stride, da_stride, du_stride;
  const void* gamma;
  const void* beta;
  float* dgamma;
  float* dbeta;
  void* workspace;
  size_t workspace_bytes;
  const void* u_pre;          /* or null.  Given: u = silu(u_pre) (and is not read), and du is the gradient of u_pre (u's, rounded, times silu') */
  int64_t u_pre_stride;
  const void* add;            /* or null.  Given: added to the rounded da (a gradient that reaches `a` another way) */
  int64_t add_stride;
  const int32_t* row_map;     /* or null.  Given: row r of dout is at row row_map[r] of its buffer */
} HstuNormGateBwdArgs;

size_t hstu_norm_gate_bwd_workspace_bytes(int64_t rows, int32_t width);
int hstu_norm_gate_bwd(const HstuNormGateBwdArgs* args, void* stream);
/* The same with dgamma and dbeta bf16 [width]: the sums rounded (the parameters' own type). */
int hstu_norm_gate_bwd_rounded(const HstuNormGateBwdArgs* args, void* stream);

/* out[m, n] = silu(sum_k x[m, k] w[k, n] + bias[n]); x: bf16 [M, K] (row stride
 * x_stride), w: bf16 [K, N] contiguous, bias: bf16 [N] or null, out: bf16
 * [M, N] contiguous; with `c` (bf16 [M, N], row stride c_stride, 16-byte aligned,
 * c_stride a multiple of 8) out = act(x w + c + bias).  fp32 accumulation, one
 * rounding.  x, w, bias, out and workspace must be 16-byte aligned and x_stride
 * a multiple of 8 elements (HSTU_BLOCK_ERR_SHAPE otherwise); N and K multiples
 * of 8 run on the matrix cores, others element by element.  `workspace` is not
 * used and may be null. */
typedef struct HstuGemmSiluArgs {
  uint32_t struct_size;   /* sizeof(HstuGemmSiluArgs)  */
  uint32_t version;       /* HSTU_BLOCK_ABI_VERSION    */
  int64_t M;
  int32_t N, K;
  int32_t activation;     /* 1: silu (the projections); 0: none */
  int32_t reserved0;
  const void* x;
  int64_t x_stride;
  const void* w;
  const void* bias;
  void* out;
  void* workspace;
  size_t workspace_bytes;
  const void* c;          /* bf16 [M, N] added to the product before bias and activation, or null: the block's */
  int64_t c_stride;       /* residual as the product's C operand (hstu.py:474), no pass of its own; row stride */
} HstuGemmSiluArgs;

size_t hstu_gemm_silu_workspace_bytes(void);
int hstu_gemm_silu_fwd(const HstuGemmSiluArgs* args, void* stream);

/* out[t, :] = gamma * (x_t - mean) * rstd + beta with x_t = scale * table[ids[t], :]
 * (+ pos_table[positions[t], :] when pos_table is given), statistics over the
 * `width` entries of x_t as in hstu_norm_gate_fwd.  table: bf16 [vocab, width]
 * (row stride table_stride), pos_table: bf16 [n_positions, width] contiguous or
 * null, ids / positions: int64 [rows] (positions null with pos_table null),
 * out: bf16 [rows, width] contiguous.  Indices outside their table are clamped
 * into it (the reference's gather on an accelerator does the same) or, with
 * `outside`, reported.  width a
 * multiple of 8 up to 8192; pointers and table_stride multiples of 8 elements. */
typedef struct HstuEmbedNormArgs {
  uint32_t struct_size;   /* sizeof(HstuEmbedNormArgs) */
  uint32_t version;       /* HSTU_BLOCK_ABI_VERSION    */
  int64_t rows;
  int32_t width;
  float eps;
  float scale;            /* 1, or sqrt(model_dim) (scale_by_sqrt_dim) */
  int32_t reserved0;
  const int64_t* ids;
  const void* table;
  int64_t vocab, table_stride;
  const int64_t* positions;
  const void* pos_table;
  int64_t n_positions;
  const void* gamma;
  const void* beta;
  void* out;
  const int32_t* row_map; /* or null.  Given: row r takes entry row_map[r] of ids (hstu_pack_plan) */
  int32_t L;              /* with positions null and pos_table given: the position is that entry's index modulo L */
  int32_t round_steps;    /* 1: the scaled row and the sum are each rounded to bf16 (what separate steps leave); 0: one rounding */
  void* sums;             /* or null (with round_steps only): x_t is stored here as well, bf16 [rows, width], for the gradients: */
                          /* hstu_norm_gate_bwd on these rows gives the gradient at x_t, whatever becomes of the tables */
  int64_t* keys;          /* or null: the row of `table` that each row took, [rows] (the keys of hstu_embed_grad) */
  int32_t* outside;       /* or null: indices are clamped.  Given (one int32 that the device can write): negative ids count from the */
                          /* table's end, and the word becomes 1 when an id or a position lies outside its table (it is clamped then) */
} HstuEmbedNormArgs;

int hstu_embed_norm_fwd(const HstuEmbedNormArgs* args, void* stream);

/* The gradient of a gathered table, all of it: out[v, :] = the sum of scale * g[t, :] over the rows t whose key is v, added in the
 * order of the rows with every term and partial sum rounded to bf16 (the bits of torch's gather backward; rows of up to 64
 * elements, and by_position = 2: partial sums in fp32); zeros for keys without a row.  The key is the id (or position) as hstu_embed_norm_fwd finds it, clamped
 * into [0, keys).  out: bf16 [keys, width] contiguous. */
typedef struct HstuEmbedGradArgs {
  uint32_t struct_size;   /* sizeof(HstuEmbedGradArgs) */
  uint32_t version;       /* HSTU_BLOCK_ABI_VERSION    */
  int64_t rows, keys;
  int32_t width;
  float scale;
  const void* g;
  int64_t g_stride;
  const int64_t* ids;
  const int64_t* positions;
  const int32_t* row_map;
  int32_t L, by_position; /* by_position 1 or 2: the keys are positions (positions, or the entry's index modulo L) */
  void* out;
  void* workspace;
  size_t workspace_bytes;
} HstuEmbedGradArgs;

size_t hstu_embed_grad_workspace_bytes(int64_t rows, int64_t keys, int32_t width);
int hstu_embed_grad(const HstuEmbedGradArgs* args, void* stream);

/* Packing a padded batch [B, L] of the given lengths (int32 or int64 [B], clamped to [0, L]): seq_offsets int32 [B + 1],
 * row_map int32 [B L] (its first *total entries: the padded row of each packed token), total: one int32 that the device can
 * write (pinned host memory will do). */
int hstu_pack_plan(const void* lens, int32_t lens_are_64bit, int32_t B, int32_t L, int32_t* seq_offsets, int32_t* row_map, int32_t* total, void* stream);
/* Lengths of an end-padded batch from its byte mask [B, L]; *bad becomes 1 when a row is not non-zero bytes followed by zeros
 * (and stays as it was otherwise). */
int hstu_mask_lengths(const uint8_t* mask, int32_t B, int32_t L, int32_t* lens, int32_t* bad, void* stream);
/* hstu_embed_norm_fwd and, with a mask, hstu_mask_lengths on it in the same launch. */
int hstu_embed_norm_mask_fwd(const HstuEmbedNormArgs* args, const uint8_t* mask, int32_t B, int32_t L, int32_t* lens, int32_t* bad, void* stream);
/* d[r, :] *= silu'(pre[r, :]) in place, bf16 rows of `width` elements. */
int hstu_silu_bwd(void* d, int64_t d_stride, const void* pre, int64_t pre_stride, int64_t rows, int32_t width, void* stream);

/* The block's matrix products without a library: bf16 operands, fp32 accumulation, one rounding.
 *   HSTU_GEMM_NN   out[M, N] = act(x[M, K] w[K, N] + c + bias)    a projection (recml/layers/keras/hstu.py:444-449, 473-474)
 *   HSTU_GEMM_NT   out[M, K] = x[M, N] w[K, N]^T                  the gradient of its input
 *   HSTU_GEMM_TN   w[K, N]   = x[M, K]^T y[M, N]                  the gradient of its weight (w written)
 * The weight comes as `slabs` matrices [K, N / slabs], contiguous each, side by side along N (the U, Q, K and V kernels
 * of a block); the other operands are single matrices with a row stride.  NN: bias [N], c [M, N] (row stride c_stride) and
 * `pre` (bf16 [M, N] contiguous: the value before the activation, which then applies to the rounded value) may be null; out is contiguous.
 * N, K, N / slabs and the row strides multiples of 8, pointers 16-byte aligned.  TN sums a long M in parts: `workspace`
 * of hstu_gemm_workspace_bytes(op, M, N, K) bytes, owned by the caller; the parts are added in a fixed order. */
#define HSTU_GEMM_NN 0
#define HSTU_GEMM_NT 1
#define HSTU_GEMM_TN 2
#define HSTU_GEMM_MAX_SLABS 4
typedef struct HstuGemmArgs {
  uint32_t struct_size;   /* sizeof(HstuGemmArgs)      */
  uint32_t version;       /* HSTU_BLOCK_ABI_VERSION    */
  int32_t op;
  int32_t activation;     /* NN: 1 = silu, 0 = none */
  int64_t M;
  int32_t N, K;
  int32_t slabs, reserved0;
  const void* x;
  int64_t x_stride;
  const void* w[HSTU_GEMM_MAX_SLABS];
  const void* y;
  int64_t y_stride;
  const void* bias;
  const void* c;
  int64_t c_stride;
  void* out;
  void* pre;
  void* workspace;
  size_t workspace_bytes;
} HstuGemmArgs;

size_t hstu_gemm_workspace_bytes(int32_t op, int64_t M, int32_t N, int32_t K);
int hstu_gemm(const HstuGemmArgs* args, void* stream);

/* The layer norm in front of a product and the product as one launch, for large batches (hstu.py:443-449): out = silu(layer_norm(x) w), the
 * normed rows rounded as hstu_norm_gate_fwd rounds them.  bf16; x [M, K] with a row stride of whole 16 bytes, gamma and beta [K], w as in
 * HstuGemmArgs, out [M, N] contiguous.  Which sizes there are: hstu_norm_gemm_takes (1 or 0). */
typedef struct HstuNormGemmArgs {
  uint32_t struct_size;   /* sizeof(HstuNormGemmArgs) */
  uint32_t version;       /* HSTU_BLOCK_ABI_VERSION   */
  int64_t M;
  int32_t N, K, slabs;
  float eps;
  const void* x;
  int64_t x_stride;
  const void* gamma;
  const void* beta;
  const void* w[HSTU_GEMM_MAX_SLABS];
  void* out;
} HstuNormGemmArgs;

int hstu_norm_gemm_takes(int64_t M, int32_t N, int32_t K, int32_t slabs);
int hstu_norm_gemm(const HstuNormGemmArgs* args, void* stream);

/* A whole block in inference as one launch, for short sequences and narrow models (hstu.py:442-474): out = tokens + output projection of
 * u * layer_norm(attention) with u, q, k, v = silu(layer_norm(tokens) w + bias), causal pointwise attention over alpha q k^T
 * (+ pos_tab) with the weights scaled by inv_n and each sequence's length.  bf16 tensors and parameters, contiguous; tokens and out
 * [B, L, width], or with seq_offsets [T, width] (sequence b from row seq_offsets[b] on, at most L rows of it).  w[i]: [width, width], the
 * U, Q, K and V kernels; w_bias[i]: [width] or all null; w_out [width, width], b_out [width] or null; pos_tab: fp32
 * [pos_heads, 2 L - 1] or null, pos_heads 1 or heads.  Which shapes there are: hstu_block_small_takes (1 or 0). */
typedef struct HstuBlockSmallArgs {
  uint32_t struct_size;   /* sizeof(HstuBlockSmallArgs) */
  uint32_t version;       /* HSTU_BLOCK_ABI_VERSION     */
  int32_t B, L, heads, head_dim, width, pos_heads;
  float eps, alpha, inv_n;
  int32_t reserved0;
  const void* tokens;
  void* out;
  const int32_t* seq_lens;
  const int32_t* seq_offsets;
  const void* in_gamma;
  const void* in_beta;
  const void* w[4];
  const void* w_bias[4];
  const void* attn_gamma;
  const void* attn_beta;
  const void* w_out;
  const void* b_out;
  const float* pos_tab;
} HstuBlockSmallArgs;

int hstu_block_small_takes(int32_t B, int32_t L, int32_t heads, int32_t head_dim, int32_t width);
int hstu_block_small_fwd(const HstuBlockSmallArgs* args, void* stream);
/* n (1 .. HSTU_BLOCK_SMALL_STACK) such blocks one behind the other in one launch: blocks[0].tokens through all of them to
 * blocks[n - 1].out (the others' tokens and out are not looked at), then, with end_gamma and end_beta [width], a layer norm of the rows
 * (hstu.py:619).  The blocks share everything but their parameters and eps. */
#define HSTU_BLOCK_SMALL_STACK 16
int hstu_block_small_stack_fwd(const HstuBlockSmallArgs* blocks, int32_t n, const void* end_gamma, const void* end_beta, float end_eps,
                               void* stream);

int hstu_block_abi_version(void);
const char* hstu_block_last_error(void);

#ifdef __cplusplus
}
#endif
#endif /* HSTU_BLOCK_H_ */
