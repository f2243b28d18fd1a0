"""HSTU block and model forward around the MI355X attention kernel.

The harness for the end-to-end (config-4) shape.  In bf16 on a GPU a block is one native call
(recml_amd/csrc/native.cpp: block) of five kernels: layer norm, the U/Q/K/V projections as one product
with their SiLU in its epilogue, the attention, its norm and the U gate in one pass, the output product
with the residual; with gradients wanted the same call records one graph node whose backward runs the
kernels' backward and writes the four slices of the projection's gradient in place.  The model's front
end (gather, position embedding, norm) and its closing norm, which also unpacks packed tokens, are one
kernel each way too.  In fp32 the steps around the attention kernels are plain torch.  A block built
with a dropout rate drops attention weights in training mode inside the attention kernels (forward and
backward regenerate the same keep pattern from a seed drawn per call), and the model drops embedding
entries with torch's dropout; in eval mode neither does anything.  Parameters are created frozen:
`requires_grad_(True)` makes them trainable.

Mirrors, name for name:
  HSTUBlock   recml/layers/keras/hstu.py:240-474 (weights :281-354, call :422-474)
  HSTU        recml/layers/keras/hstu.py:492-621 (call :585-621)

Differences from the reference layer, on purpose:
  * the [B, L, L] attention mask and bias tensors are never built: the block
    takes `seq_lens` (end-padded batches, as the reference's data pipeline
    produces) and the bias *tables* (`pos_bias`, `timestamps` + `ts_bias`);
  * U, Q, K, V come from one [D, 4D] product over the four kernels, which are stored
    separately under the reference's names;
  * softmax attention (hstu.py:392-420) is not implemented here.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from recml_amd import _native
from recml_amd import hstu_block_ops
from recml_amd import hstu_ops
from recml_amd import masks


def _wants_grad(*tensors) -> bool:
  return torch.is_grad_enabled() and any(isinstance(t, torch.Tensor) and t.requires_grad for t in tensors)


def _differentiates(*tensors) -> bool:
  """Whether a gradient is asked for in either mode."""
  return _wants_grad(*tensors) or _native.has_tangent(*tensors)


def _ready(t, dtype):
  """A lengths, timestamps or table tensor as the kernels read it."""
  return t if not isinstance(t, torch.Tensor) or (t.dtype == dtype and t.is_contiguous()) else t.to(dtype).contiguous()


def _attention(q, k, v, *, pos_bias=None, ts_bias=None, batch=None, **kw):
  """The attention op, differentiable when anything it reads wants a gradient: through the HIP
  backward kernels for q, k, v, the bias tables and a dense bias.  `batch`: the per-batch preparation
  shared by the layers (inference only)."""
  if _differentiates(q, k, v, pos_bias, ts_bias, kw.get("bias")):
    return hstu_ops.hstu_attention_autograd(q, k, v, pos_bias=pos_bias, ts_bias=ts_bias, **kw)
  return hstu_ops.hstu_attention(q, k, v, pos_bias=pos_bias, ts_bias=ts_bias, batch=batch, **kw)


class _AttentionGateFn(torch.autograd.Function):
  """gated = u * layer_norm(attention(q, k, v)) on the four slices of ONE projection uqkv [..., 4, H, hd]
  (contiguous, bf16), with every gradient through the HIP kernels, which write dq, dk, dv and du straight
  into the slices of one gradient tensor shaped like the projection."""

  @staticmethod
  def forward(ctx, uqkv, gamma, beta, pos_bias, ts_bias, eps, batch, kwargs):
    uqkv = uqkv.contiguous()            # (the backward mirrors this layout for the gradient)
    u, q, k, v = uqkv.unbind(dim=-3)
    attn = hstu_ops.hstu_attention(q, k, v, pos_bias=pos_bias, ts_bias=ts_bias, batch=batch, **kwargs)
    W = q.shape[-2] * q.shape[-1]
    gated = hstu_block_ops.norm_gate(attn.reshape(-1, W).detach(), u.reshape(-1, W).detach(), gamma.detach().reshape(-1),
                                     beta.detach().reshape(-1), eps)
    ctx.save_for_backward(uqkv, attn, gamma, beta, *(t for t in (pos_bias, ts_bias) if t is not None))
    ctx.has = (pos_bias is not None, ts_bias is not None)
    ctx.eps, ctx.kwargs = eps, kwargs
    return gated.reshape(*uqkv.shape[:-3], W)

  @staticmethod
  def backward(ctx, dgated):
    uqkv, attn, gamma, beta, *rest = ctx.saved_tensors
    pos = rest.pop(0) if ctx.has[0] else None
    ts = rest.pop(0) if ctx.has[1] else None
    u, q, k, v = uqkv.unbind(dim=-3)
    W = q.shape[-2] * q.shape[-1]
    d_uqkv = torch.empty_like(uqkv)                     # uqkv is contiguous: the same strides
    du, dq, dk, dv = d_uqkv.unbind(dim=-3)
    du2 = du.reshape(-1, W)
    assert du2.data_ptr() == du.data_ptr()              # a view: the kernel writes into d_uqkv
    d_attn, _, dg, db = hstu_block_ops.norm_gate_bwd(attn.reshape(-1, W), u.reshape(-1, W), gamma.reshape(-1), beta.reshape(-1),
                                                     dgated.reshape(-1, W).contiguous(), ctx.eps, du_out=du2)
    # needs_input_grad follows forward's arguments: uqkv, gamma, beta, pos_bias, ts_bias, ...
    want_tables = (pos is not None and ctx.needs_input_grad[3]) or (ts is not None and ctx.needs_input_grad[4])
    _, _, _, dpos, dts = hstu_ops.hstu_attention_bwd(q, k, v, d_attn.reshape(attn.shape), pos_bias=pos, ts_bias=ts,
                                                     table_grads=want_tables, grads_out=(dq, dk, dv), **ctx.kwargs)
    cast = lambda g, t: None if g is None else g.to(t.dtype)
    return (d_uqkv, dg.to(gamma.dtype).reshape(gamma.shape), db.to(beta.dtype).reshape(beta.shape),
            cast(dpos, pos) if pos is not None else None, cast(dts, ts) if ts is not None else None, None, None, None)


class _OutputProjectionFn(torch.autograd.Function):
  """gated @ W (+ bias) + residual with the residual as the product's C operand (recml/layers/keras/hstu.py:473-474):
  torch's addmm copies the residual into the output before the product.  The gradients are two plain products."""

  @staticmethod
  def forward(ctx, gated, w, bias, residual):
    ctx.save_for_backward(gated, w)
    ctx.has_bias = bias is not None
    return hstu_block_ops.gemm_silu(gated, w, bias, False, residual=residual)

  @staticmethod
  def backward(ctx, dout):
    gated, w = ctx.saved_tensors
    need = ctx.needs_input_grad
    d_gated = dout @ w.t() if need[0] else None
    d_w = gated.t() @ dout if need[1] else None
    d_bias = dout.sum(0) if (ctx.has_bias and need[2]) else None
    return d_gated, d_w, d_bias, dout if need[3] else None


def _glorot_uniform(shape, fan_in, fan_out, generator, dtype, device):
  limit = math.sqrt(6.0 / (fan_in + fan_out))
  w = torch.empty(shape, dtype=torch.float32)
  w.uniform_(-limit, limit, generator=generator)
  return w.to(device=device, dtype=dtype)


class HSTUBlock(torch.nn.Module):
  """One HSTU block: LN -> U,Q,K,V = act(x W) -> pointwise attention -> LN over
  (heads, head_dim) -> U * normed -> output projection -> + inputs
  (recml/layers/keras/hstu.py:444-474)."""

  def __init__(self, hidden_dim: int, num_heads: int, use_bias: bool = False,
               layer_norm_epsilon: float = 1e-6, scaled_pointwise_attn: bool = False,
               softmax_attention: bool = False, dropout: float = 0.0,
               dtype=torch.float32, device=None, generator=None):
    super().__init__()
    if softmax_attention:
      raise NotImplementedError("softmax attention is outside this build; only the pointwise path is accelerated")
    if hidden_dim % num_heads:
      raise ValueError(f"hidden_dim {hidden_dim} is not a multiple of num_heads {num_heads}")
    if not 0.0 <= dropout < 1.0:
      raise ValueError(f"dropout must be in [0, 1), got {dropout}")
    # The reference drops attention weights in training (recml/layers/keras/hstu.py:386-387): here the attention
    # kernels do it, from a seed this block draws per forward.
    self.dropout = float(dropout)
    self.num_heads = num_heads
    self.head_dim = hidden_dim // num_heads
    self.hidden_dim = hidden_dim
    self.eps = layer_norm_epsilon
    self.scaled_pointwise_attn = scaled_pointwise_attn
    H, hd, D = num_heads, self.head_dim, hidden_dim
    P = torch.nn.Parameter
    # EinsumDense "btd,dnh->btnh": kernel [D, H, hd], Glorot-uniform with the fans Keras
    # computes for a rank-3 shape (see _fans)
    fi, fo = self._fans((D, H, hd))
    for name in ("u", "q", "k", "v"):
      self.register_parameter(f"{name}_kernel", P(_glorot_uniform((D, H, hd), fi, fo, generator, dtype, device), requires_grad=False))
      if use_bias:
        self.register_parameter(f"{name}_bias", P(torch.zeros((H, hd), dtype=dtype, device=device), requires_grad=False))
    fi, fo = self._fans((H, hd, D))
    self.output_kernel = P(_glorot_uniform((H, hd, D), fi, fo, generator, dtype, device), requires_grad=False)
    self.output_bias = P(torch.zeros((D,), dtype=dtype, device=device), requires_grad=False) if use_bias else None
    self.use_bias = use_bias
    self.input_ln_gamma = P(torch.ones((D,), dtype=dtype, device=device), requires_grad=False)
    self.input_ln_beta = P(torch.zeros((D,), dtype=dtype, device=device), requires_grad=False)
    self.attn_ln_gamma = P(torch.ones((H, hd), dtype=dtype, device=device), requires_grad=False)
    self.attn_ln_beta = P(torch.zeros((H, hd), dtype=dtype, device=device), requires_grad=False)

  @staticmethod
  def _fans(shape):
    """Keras' fan computation for a rank-3 kernel: the leading axes are the
    receptive field (keras/src/initializers/random_initializers.py,
    compute_fans): fan_in = shape[-2] * prod(shape[:-2]), fan_out = shape[-1] * prod(shape[:-2])."""
    rf = 1
    for s in shape[:-2]:
      rf *= s
    return shape[-2] * rf, shape[-1] * rf

  def _dropout_kw(self, dropout_seed=None) -> dict:
    """The attention's dropout arguments for this call: none in eval mode or at rate 0; in training mode the
    block's rate and a seed from torch's CPU generator (so torch.manual_seed makes a run repeatable, and no GPU
    work waits on it) unless the caller brings one."""
    if not (self.training and self.dropout > 0.0):
      return {}
    if dropout_seed is None:
      dropout_seed = int(torch.randint(0, 2 ** 62, (1,)).item())
    return dict(dropout_p=self.dropout, dropout_seed=int(dropout_seed))

  def forward(self, inputs, *, seq_lens=None, pos_bias=None, timestamps=None, ts_bias=None,
              attention_mask=None, attention_bias=None, batch=None, dropout_seed=None):
    """inputs [B, L, D] -> [B, L, D].

    Give `seq_lens` [B] (keys and rows at or past the length are masked, as
    make_causal_mask does for an end-padded batch) with optional bias tables;
    or, for the reference's calling convention, a dense `attention_mask`
    [B, L, L] and optional `attention_bias` [B, L, L]
    (recml/layers/keras/hstu.py:422-440), beside which lengths and tables are not looked at.  `batch`: an `hstu_ops.AttentionBatch` shared with the
    other blocks that see the same lengths, timestamps and tables.  `dropout_seed`: in training mode
    with a dropout rate, the seed of this call's keep pattern (default: drawn from torch's generator).
    """
    drop = self._dropout_kw(dropout_seed)
    B, L, D = inputs.shape
    H, hd = self.num_heads, self.head_dim
    if attention_mask is not None:
      # the mask stands in place of the lengths, and the dense bias in place of the tables (hstu.py:422-440)
      seq_lens = pos_bias = timestamps = ts_bias = None
    out = self._native_steps(inputs, L, batch, drop, pos_bias, timestamps, ts_bias, seq_lens=seq_lens,
                             attention_mask=attention_mask, attention_bias=attention_bias)
    if out is not None:
      return out
    alpha, n = self._alpha_n(L)
    if attention_mask is None and attention_bias is None and self._fused_training(inputs, pos_bias, ts_bias):
      return self._train_steps(inputs.reshape(B * L, D), (B, L), pos_bias, ts_bias, batch,
                               dict(seq_lens=seq_lens, n=n, alpha=alpha, timestamps=timestamps, **drop)).reshape(B, L, D)
    fused = self._fused_inference(inputs, pos_bias, ts_bias, attention_bias)
    u, q, k, v = self._project(self._input_norm(inputs, fused).reshape(B * L, D), (B, L), fused).unbind(dim=2)
    if attention_mask is not None:
      # the reference's calling convention: a dense [B, L, L] mask and bias (training: forward and backward kernels,
      # the gradient of a dense bias included)
      attn = hstu_ops.pointwise_attention(q, k, v, attention_mask, attention_bias,
                                          scaled_pointwise_attn=self.scaled_pointwise_attn, batch=batch, **drop)
    else:
      attn = _attention(q, k, v, seq_lens=seq_lens, n=n, alpha=alpha, pos_bias=pos_bias,
                        timestamps=timestamps, ts_bias=ts_bias, bias=attention_bias, batch=batch, **drop)
    return self._gate_and_output(attn.reshape(B * L, H * hd), u.reshape(B * L, H * hd), inputs.reshape(B * L, D), fused).reshape(B, L, D)

  def _alpha_n(self, L):
    """The logit scale and the normaliser (recml/layers/keras/hstu.py:365-378)."""
    return (1.0 / math.sqrt(self.head_dim), 1.0) if self.scaled_pointwise_attn else (1.0, float(L))

  def _input_norm(self, t, fused):
    if fused:
      return hstu_block_ops.layer_norm(t, self.input_ln_gamma, self.input_ln_beta, self.eps)
    return F.layer_norm(t, (self.hidden_dim,), self.input_ln_gamma, self.input_ln_beta, self.eps)

  def _project(self, x, lead, fused):
    """U, Q, K, V of normalised rows: [*lead, 4, H, hd].  `fused`: the activation in the product's epilogue."""
    w, b = self._uqkv_weights()
    if fused:
      uqkv = hstu_block_ops.gemm_silu(x, w, b, True)
    else:
      uqkv = x @ w
      uqkv = F.silu(uqkv if b is None else uqkv + b)
    return uqkv.reshape(*lead, 4, self.num_heads, self.head_dim)

  def _gate_and_output(self, attn, u, residual, fused):
    """Attention norm, U gate, output product and residual, on rows.  `fused`: norm and gate in one pass, rounded once, and the
    residual as the product's C operand."""
    W = attn.shape[-1]
    gamma, beta, w = self.attn_ln_gamma.reshape(-1), self.attn_ln_beta.reshape(-1), self.output_kernel.reshape(W, self.hidden_dim)
    if fused:
      return hstu_block_ops.gemm_silu(hstu_block_ops.norm_gate(attn, u, gamma, beta, self.eps), w, self.output_bias, False, residual=residual)
    out = (u * F.layer_norm(attn, (W,), gamma, beta, self.eps)) @ w
    if self.use_bias:
      out = out + self.output_bias
    return out + residual

  def _weights(self):
    """The block's parameters as the native call takes them: whatever stands under their names (a parametrization or a pruning mask
    puts a tensor of its own there)."""
    P = self._parameters                 # (a module's attribute lookup costs four times the dictionary's)
    try:
      if not self.use_bias:
        return (P["input_ln_gamma"], P["input_ln_beta"], P["u_kernel"], P["q_kernel"], P["k_kernel"], P["v_kernel"], None, None, None, None,
                P["attn_ln_gamma"], P["attn_ln_beta"], P["output_kernel"], None)
      return (P["input_ln_gamma"], P["input_ln_beta"], P["u_kernel"], P["q_kernel"], P["k_kernel"], P["v_kernel"], P["u_bias"], P["q_bias"],
              P["k_bias"], P["v_bias"], P["attn_ln_gamma"], P["attn_ln_beta"], P["output_kernel"], P["output_bias"])
    except KeyError:
      biases = (self.u_bias, self.q_bias, self.k_bias, self.v_bias) if self.use_bias else (None,) * 4
      return (self.input_ln_gamma, self.input_ln_beta, self.u_kernel, self.q_kernel, self.k_kernel, self.v_kernel, *biases,
              self.attn_ln_gamma, self.attn_ln_beta, self.output_kernel, self.output_bias if self.use_bias else None)

  def _wants_grad(self, *tensors) -> bool:
    return _differentiates(*self._weights(), *tensors)

  def _fused_inference(self, t, *bias_inputs) -> bool:
    """Whether the steps of hstu_block_ops apply where the native call does not: bf16 on a GPU, nothing asking for gradients, widths
    the norm kernels take."""
    D = self.hidden_dim
    return t.is_cuda and t.dtype == torch.bfloat16 and D % 8 == 0 and D <= 8192 and not self._wants_grad(t, *bias_inputs)

  def _fused_training(self, t, *bias_inputs) -> bool:
    """Whether the training form of the fused steps (native, or _train_steps) applies: bf16 on a GPU, something asking for a gradient,
    widths the norm kernels' backward takes."""
    D, W = self.hidden_dim, self.num_heads * self.head_dim
    return (t.is_cuda and t.dtype == torch.bfloat16 and self._wants_grad(t, *bias_inputs)
            and D % 8 == 0 and W % 8 == 0 and D <= 2048 and W <= 2048)

  def _train_steps(self, tokens, lead, pos_bias, ts_bias, batch, attn_kw):
    """The block on rows [T, D] with gradients where the native call does not apply (head dims or parameters that are not laid out for
    it): norms, attention and gate through the HIP kernels, the products and the projections' SiLU in torch.  `lead`: the leading
    shape of the attention's tensors ((B, L) padded, (T,) packed)."""
    x = hstu_block_ops.layer_norm(tokens, self.input_ln_gamma, self.input_ln_beta, self.eps)
    uqkv = self._project(x, lead, False)
    gated = _AttentionGateFn.apply(uqkv, self.attn_ln_gamma, self.attn_ln_beta, pos_bias, ts_bias, self.eps, batch, attn_kw)
    W = self.num_heads * self.head_dim
    return _OutputProjectionFn.apply(gated.reshape(-1, W), self.output_kernel.reshape(W, self.hidden_dim), self.output_bias, tokens)

  def _native_steps(self, tokens, length, batch, drop, pos_bias, timestamps, ts_bias, seq_lens=None, seq_offsets=None,
                    attention_mask=None, attention_bias=None):
    """The block through its HIP kernels, forward and backward, as one native call (recml_amd/csrc/native.cpp: block): bf16 on a
    GPU, parameters ready as they are.  None where it does not apply: fp32, a dense mask or bias with gradients, ..."""
    if tokens.dtype != torch.bfloat16 or not tokens.is_cuda:
      return None
    weights = self._weights()
    grad = _wants_grad(tokens, *weights, pos_bias, ts_bias, attention_bias)
    if grad and not (self._fused_training(tokens, pos_bias, ts_bias) and hstu_ops.hstu_attention_bwd is hstu_ops._OWN_ATTENTION_BWD
                     and hstu_block_ops.norm_gate_bwd is hstu_block_ops._OWN_NORM_GATE_BWD):
      return None
    alpha, n = self._alpha_n(length)
    got = _native.block(tokens.contiguous(), weights, self.num_heads, self.head_dim, self.eps, alpha, n, seq_lens, seq_offsets,
                        None if seq_offsets is None else length, pos_bias, timestamps, ts_bias, attention_mask, attention_bias,
                        drop.get("dropout_p", 0.0), drop.get("dropout_seed", 0),
                        False if batch is None else batch._prepared, None if batch is None else batch._buf, grad)
    if got is None:
      # (declined before any work.  torch's default integers, 16-bit tables: converted, by the first block of a batch for all of them; a
      # table's conversion is part of the graph)
      ready = _ready if batch is None else batch.ready
      table = _ready if grad else ready
      given = seq_lens, seq_offsets, timestamps, pos_bias, ts_bias
      seq_lens, seq_offsets, timestamps = ready(seq_lens, torch.int32), ready(seq_offsets, torch.int32), ready(timestamps, torch.int64)
      pos_bias, ts_bias = table(pos_bias, torch.float32), table(ts_bias, torch.float32)
      if all(x is y for x, y in zip(given, (seq_lens, seq_offsets, timestamps, pos_bias, ts_bias))):
        return None
      return self._native_steps(tokens, length, batch, drop, pos_bias, timestamps, ts_bias, seq_lens, seq_offsets, attention_mask,
                                attention_bias)
    out, signature, workspace, reused = got
    if batch is not None:
      batch._keep_native(signature, workspace, reused, (seq_lens, seq_offsets, timestamps, pos_bias, ts_bias, attention_mask))
    return out

  def _uqkv_weights(self):
    w = torch.cat([self.u_kernel, self.q_kernel, self.k_kernel, self.v_kernel], dim=1).reshape(self.hidden_dim, -1)
    b = torch.cat([self.u_bias, self.q_bias, self.k_bias, self.v_bias], dim=0).reshape(-1) if self.use_bias else None
    return w, b

  def forward_jagged(self, tokens, seq_offsets, max_len, *, pos_bias=None, timestamps=None, ts_bias=None, batch=None,
                     dropout_seed=None):
    """The block on packed tokens [T, D] (sequence b = rows seq_offsets[b]..seq_offsets[b+1]):
    no work at all for padding, in the projections either.  `timestamps` is jagged [T].

    In bf16 the steps run fused: the projections' SiLU in the epilogue of their one matrix product, the
    attention norm and the U gate in one pass, the residual added by the output product."""
    drop = self._dropout_kw(dropout_seed)
    T, D = tokens.shape
    H, hd = self.num_heads, self.head_dim
    out = self._native_steps(tokens, int(max_len), batch, drop, pos_bias, timestamps, ts_bias, seq_offsets=seq_offsets)
    if out is not None:
      return out
    alpha, n = self._alpha_n(max_len)
    if self._fused_training(tokens, pos_bias, ts_bias):
      return self._train_steps(tokens, (T,), pos_bias, ts_bias, batch,
                               dict(seq_offsets=seq_offsets, max_len=max_len, n=n, alpha=alpha, timestamps=timestamps, **drop))
    fused = self._fused_inference(tokens, pos_bias, ts_bias)
    u, q, k, v = self._project(self._input_norm(tokens, fused), (T,), fused).unbind(dim=1)
    attn = _attention(q, k, v, seq_offsets=seq_offsets, max_len=max_len, n=n, alpha=alpha,
                      pos_bias=pos_bias, timestamps=timestamps, ts_bias=ts_bias, batch=batch, **drop)
    return self._gate_and_output(attn.reshape(T, H * hd), u.reshape(T, H * hd), tokens, fused)


_OWN_BLOCK_FORWARDS = HSTUBlock.forward, HSTUBlock.forward_jagged


def _is_plain_call(block, jagged) -> bool:
  """Whether a call of the block is a call of HSTUBlock's own forward and nothing else: no subclass, no forward put in its place, and, where
  it is called as a module (the packed form calls forward_jagged itself), no hooks on it or on all modules, and not compiled."""
  if type(block) is not HSTUBlock or (HSTUBlock.forward, HSTUBlock.forward_jagged) != _OWN_BLOCK_FORWARDS:
    return False
  own = block.__dict__
  if jagged:
    return "forward_jagged" not in own
  m = torch.nn.modules.module
  return ("forward" not in own and block._compiled_call_impl is None
          and not (own["_forward_hooks"] or own["_forward_pre_hooks"] or own["_backward_hooks"] or own["_backward_pre_hooks"]
                   or m._global_forward_hooks or m._global_forward_pre_hooks or m._global_backward_hooks or m._global_backward_pre_hooks))


class HSTU(torch.nn.Module):
  """The HSTU model forward (recml/layers/keras/hstu.py:585-621): item
  embedding (x sqrt(D)) + position embedding -> final_norm -> blocks ->
  final_norm (the same layer both times) -> optional untied output head."""

  def __init__(self, *, vocab_size: int, max_positions: int | None = None, model_dim: int,
               num_heads: int, num_layers: int, dropout: float = 0.0, norm_eps: float = 1e-6,
               scale_by_sqrt_dim: bool = False, add_head: bool = True,
               dtype=torch.float32, device=None, seed: int = 0):
    super().__init__()
    g = torch.Generator().manual_seed(seed)
    P = torch.nn.Parameter
    normal = lambda shape: (torch.randn(shape, generator=g) * 0.02).to(device=device, dtype=dtype)
    self.item_embedding = P(normal((vocab_size, model_dim)), requires_grad=False)
    self.position_embedding = P(normal((max_positions, model_dim)), requires_grad=False) if max_positions else None
    self.decoder_blocks = torch.nn.ModuleList(
        HSTUBlock(model_dim, num_heads, layer_norm_epsilon=norm_eps, dropout=dropout, dtype=dtype, device=device, generator=g)
        for _ in range(num_layers))
    self.final_norm_gamma = P(torch.ones((model_dim,), dtype=dtype, device=device), requires_grad=False)
    self.final_norm_beta = P(torch.zeros((model_dim,), dtype=dtype, device=device), requires_grad=False)
    self.reverse_embedding = P(normal((model_dim, vocab_size)), requires_grad=False) if add_head else None
    self.model_dim = model_dim
    self.eps = norm_eps
    self.scale_by_sqrt_dim = scale_by_sqrt_dim
    self.dropout = float(dropout)      # on the embeddings here (hstu.py:541-543, 602), on the attention weights in the blocks

  def count_params(self) -> int:
    return sum(p.numel() for p in self.parameters())

  def _final_norm(self, x):
    out = _native.final_norm(x, self.final_norm_gamma, self.final_norm_beta, self.eps, None, None, 0, 0, True)
    if out is not None:
      return out
    D = self.model_dim
    training = _differentiates(x, self.final_norm_gamma, self.final_norm_beta)
    if x.is_cuda and x.dtype == torch.bfloat16 and D % 8 == 0 and D <= (2048 if training else 8192):
      return hstu_block_ops.layer_norm(x, self.final_norm_gamma, self.final_norm_beta, self.eps)
    return F.layer_norm(x, (D,), self.final_norm_gamma, self.final_norm_beta, self.eps)

  def _embed(self, ids, row_map, tokens, mask):
    return _native.embed(ids if ids.dtype == torch.int64 and ids.is_contiguous() else ids.to(torch.int64).contiguous(), self.item_embedding,
                         self.position_embedding, self.final_norm_gamma, self.final_norm_beta, self.eps,
                         self.model_dim ** 0.5 if self.scale_by_sqrt_dim else 1.0, row_map, tokens, True, mask)

  def _front_end(self, ids, row_map=None, tokens=0):
    """Gather, scale, position embedding and final_norm (hstu.py:593-601): in bf16 on a GPU one pass, and one each for the
    gradients of the norm and of the tables.  ids [B, L]; the packed form with `row_map` (its `tokens` first entries).
    Returns the rows and, with gradients, a ticket for _check_indices."""
    table, positions = self.item_embedding, self.position_embedding
    scale, length = self.model_dim ** 0.5 if self.scale_by_sqrt_dim else 1.0, ids.shape[1]
    got = self._embed(ids, row_map, tokens, None)
    x, ticket = (None, None) if got is None else got
    if x is None:
      where = None if row_map is None else row_map[:tokens].to(torch.int64)
      ids = ids if where is None else ids.reshape(-1)[where]
      if table.is_cuda and table.dtype == torch.bfloat16 and not _differentiates(table, positions, self.final_norm_gamma,
                                                                                              self.final_norm_beta):
        at = None
        if positions is not None:
          at = torch.arange(length, device=ids.device).expand(ids.shape).contiguous() if where is None else where % length
        x = hstu_block_ops.embed_norm(ids.to(torch.int64), table, self.final_norm_gamma, self.final_norm_beta, self.eps, scale=scale,
                                      positions=at, pos_table=positions)
      else:
        x = table[ids]
        if self.scale_by_sqrt_dim:
          x = x * scale
        if positions is not None:
          x = x + (positions[:length] if where is None else positions[where % length])
        x = self._final_norm(x)
    return (F.dropout(x, self.dropout, self.training) if self.training and self.dropout > 0.0 else x), ticket

  def _check_indices(self, ticket):
    """Raises where the front end met an id outside the vocabulary or a position past the table (in training; inference clamps them).
    Asked when the rest of the forward is enqueued: the answer is there by then."""
    if ticket is not None and _native.raised(ticket):
      raise IndexError(f"an item id lies outside the vocabulary of {self.item_embedding.shape[0]}"
                       + ("" if self.position_embedding is None else f", or a position past the {self.position_embedding.shape[0]} there are"))

  def _narrow_blocks(self, x, length, seq_lens, offsets, pos_bias, close):
    """All blocks on x in one launch (recml_amd/csrc/hstu_block_small.hip), with `close` the closing norm behind them: narrow models in
    inference on short sequences.  None where there is no such launch, or where somebody watches or changes the blocks' calls."""
    if self.model_dim > 64 or not x.is_cuda or x.dtype != torch.bfloat16:
      return None
    blocks = self.decoder_blocks._modules.values()
    first = next(iter(blocks), None)
    if first is None or (close and type(self)._final_norm is not HSTU._final_norm):
      return None
    weights, like = [], None
    for block in blocks:
      if not _is_plain_call(block, offsets is not None) or (block.training and block.dropout > 0.0):
        return None
      kind = block.num_heads, block.head_dim, block.eps, block.scaled_pointwise_attn
      if like is not None and kind != like:
        return None
      like = kind
      weights.append(block._weights())
    alpha, n = first._alpha_n(length)
    gamma, beta = (self.final_norm_gamma, self.final_norm_beta) if close else (None, None)
    return _native.blocks(x.contiguous(), tuple(weights), first.num_heads, first.head_dim, first.eps, alpha, n, seq_lens, offsets,
                          None if offsets is None else length, pos_bias, gamma, beta, self.eps)

  def _head(self, x):
    out = _native.linear(x, self.reverse_embedding, True)
    return x @ self.reverse_embedding if out is None else out

  def forward(self, inputs, padding_mask=None, attention_mask=None, *, seq_lens=None, pos_bias=None, timestamps=None,
              ts_bias=None, jagged=False):
    """inputs: item ids [B, L]; `padding_mask` [B, L] (1 = real item, end-padded) or `seq_lens` [B]; or, as
    the reference's call also allows (hstu.py:585-615), a dense `attention_mask` [B, L, L] that every block
    then takes as it is (any mask, at the price of reading it in every layer).

    jagged=True packs the valid tokens once and runs every block on [T, D]: nothing is computed
    for padding.  Rows past a sequence's length are then returned as zeros, whereas the padded
    form (like the reference) carries the padded positions' own embeddings through the blocks.
    """
    ticket = front = None
    if attention_mask is not None:
      if jagged or pos_bias is not None or ts_bias is not None or seq_lens is not None:
        raise ValueError("`attention_mask` goes with the padded form and without `seq_lens` and bias tables")
      if isinstance(attention_mask, torch.Tensor) and attention_mask.dtype not in (torch.bool, torch.uint8):
        attention_mask = attention_mask != 0           # as the attention takes it, once for all blocks
    elif seq_lens is None:
      if padding_mask is None:
        raise ValueError("Either `attention_mask`, `padding_mask` or `seq_lens` must be set.")
      # Whether the mask is end-padded is known once its kernel has run (`ticket`).  It is asked before anything random is drawn, in the
      # packed form behind the packing's own wait, and otherwise when the first block is enqueued: the answer is there by then, where
      # waiting for it first leaves a small batch's GPU idle (32 x 50 x 64, 4 blocks: 164 us a call, 133 this way).
      # (Nothing random to draw and no packing: the lengths come with the front end, in its launch; 53.3 us a call of that size -> 50.4.)
      if not jagged and not (self.training and self.dropout > 0.0) and type(self)._front_end is HSTU._front_end:
        front = self._embed(inputs, None, 0, padding_mask)
      if front is not None:
        *front, seq_lens, ticket = front
      else:
        got = _native.mask_lengths(padding_mask)
        seq_lens, ticket = got if got is not None else (masks.lengths_from_padding_mask(padding_mask), None)
    if jagged:
      return self._forward_jagged(inputs, seq_lens, pos_bias, timestamps, ts_bias, ticket)
    if self.training and self.dropout > 0.0:
      ticket = self._check_mask(ticket)
    x, outside = self._front_end(inputs) if front is None else front
    out = None
    if attention_mask is None and timestamps is None and ts_bias is None:
      out = self._narrow_blocks(x, x.shape[1], seq_lens, None, pos_bias, True)
    if out is None:
      # every block sees the same lengths, timestamps and tables: the attention prepares them once
      batch = hstu_ops.AttentionBatch()
      for block in self.decoder_blocks:
        if attention_mask is not None:
          x = block(x, attention_mask=attention_mask, batch=batch)
        else:
          x = block(x, seq_lens=seq_lens, pos_bias=pos_bias, timestamps=timestamps, ts_bias=ts_bias, batch=batch)
        if ticket is not None:
          ticket = self._check_mask(ticket)
      out = self._final_norm(x)
    elif ticket is not None:
      ticket = self._check_mask(ticket)
    if self.reverse_embedding is not None:
      out = self._head(out)
    self._check_mask(ticket)
    self._check_indices(outside)
    return out

  def _check_mask(self, ticket):
    """Raises where the padding mask behind the ticket was not end-padded; there is nothing left to ask afterwards."""
    if ticket is not None and _native.raised(ticket):
      raise ValueError(masks.NOT_END_PADDED)

  def _forward_jagged(self, inputs, seq_lens, pos_bias, timestamps, ts_bias, ticket):
    B, L = inputs.shape
    # which padded row each packed token comes from: found once (the one host wait of the packing: the token count) and used for
    # every gather and for the scatter at the end
    # (lengths of another batch size are not for the kernels: torch's shape checks below report them)
    got = _native.pack(seq_lens, L) if seq_lens.shape == (B,) else None
    if got is None:
      lens = seq_lens.to(torch.int64).clamp(0, L)
      valid = torch.arange(L, device=inputs.device)[None, :] < lens[:, None]          # [B, L]
      offsets = torch.zeros(B + 1, dtype=torch.int32, device=inputs.device)
      offsets[1:] = torch.cumsum(lens, 0)
      rows = valid.reshape(-1).nonzero().squeeze(1).to(torch.int32)
      tokens = rows.numel()
    else:
      offsets, rows, tokens = got
    self._check_mask(ticket)
    x, outside = self._front_end(inputs, rows, tokens)
    ts = None if timestamps is None else timestamps.reshape(-1).index_select(0, rows[:tokens])
    narrow = self._narrow_blocks(x, L, None, offsets, pos_bias, False) if ts is None and ts_bias is None else None
    batch = hstu_ops.AttentionBatch()
    for block in self.decoder_blocks if narrow is None else ():
      x = block.forward_jagged(x, offsets, L, pos_bias=pos_bias, timestamps=ts, ts_bias=ts_bias, batch=batch)
    x = x if narrow is None else narrow
    if self.reverse_embedding is None:
      out = _native.final_norm(x, self.final_norm_gamma, self.final_norm_beta, self.eps, offsets, rows, B, L, True)
      if out is not None:
        self._check_indices(outside)
        return out
    x = self._final_norm(x)
    if self.reverse_embedding is not None:
      x = self._head(x)
    self._check_indices(outside)
    out = torch.zeros((B * L, x.shape[-1]), dtype=x.dtype, device=x.device)
    return out.index_copy(0, rows[:tokens].to(torch.int64), x).reshape(B, L, x.shape[-1])
