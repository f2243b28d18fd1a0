"""Dense masks and biases whose rows are no whole 16-byte pieces, in bf16 on the matrix-core kernels.

The host side gives such a matrix longer rows (hstu_attn_pad_rows) when that is all that keeps a call off the matrix-core
kernels; lengths around the kernels' tiles (32 keys, 128 rows) and around the pieces (4 floats, 16 mask bytes)."""

import numpy as np
import pytest
import torch

import recml_amd
from oracle import hstu_oracle as O

pytestmark = pytest.mark.gpu
bf = torch.bfloat16


def _dev(x, dtype=None):
  t = torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")
  return t if dtype is None else t.to(dtype)


def _rel(a, b):
  return np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)


@pytest.mark.parametrize("L", [1, 15, 33, 127, 131, 248, 302])
@pytest.mark.parametrize("d,with_mask,with_bias,shared", [(64, True, True, False), (32, True, False, True), (128, False, True, False), (128, True, True, True)])
def test_dense_rows_of_any_length(gpu, L, d, with_mask, with_bias, shared):
  rng = np.random.default_rng(100 * L + d)
  B, H = 2, 2
  q, k, v, dout = (O.round_bf16(rng.standard_normal((B, L, H, d)).astype(np.float32) * 0.4) for _ in range(4))
  nb = 1 if shared else B
  mask = (rng.random((nb, L, L)) > 0.3) & (np.arange(L)[None, None, :] <= np.arange(L)[None, :, None]) if with_mask else None
  if mask is not None and shared:
    mask = mask[0]
  bias = (rng.standard_normal((nb, L, L)) * 0.4).astype(np.float32) if with_bias else None
  kw = dict(n=float(L), alpha=0.3, causal=not with_mask)
  ref = O.hstu_attention_ref(q, k, v, mask=mask, bias=bias, **kw)
  want = O.hstu_attention_bwd_ref(q, k, v, dout, mask=mask, bias=bias, bias_grad=with_bias, **kw)
  gk = dict(kw, mask=None if mask is None else _dev(mask))
  bt = None if bias is None else _dev(bias).requires_grad_(True)
  ts = [_dev(x, bf).requires_grad_(True) for x in (q, k, v)]
  out = recml_amd.hstu_attention_autograd(*ts, bias=bt, **gk)
  out.backward(_dev(dout, bf))
  variant = []
  again = recml_amd.hstu_attention_bwd(*(t.detach() for t in ts), _dev(dout, bf), bias=None if bt is None else bt.detach(), bias_grad=with_bias,
                                       _variant_out=variant, **gk)
  torch.cuda.synchronize()
  assert variant == ["hstu_bwd_mfma_bf16"]
  assert _rel(out.detach().float().cpu().numpy(), ref) <= 2e-2
  for nm, t, g, w in zip(("dq", "dk", "dv"), ts, again[:3], want[:3]):
    assert torch.equal(t.grad, g), nm                      # both host sides, the same kernels
    assert _rel(g.float().cpu().numpy(), w) <= 2e-2, nm
  if with_bias:
    assert _rel(bt.grad.cpu().numpy(), want[5]) <= 2e-2


def _beside(x):
  """The same values in rows that are no whole 16 bytes apart: such a call is the general kernel's."""
  B, L, H, d = x.shape
  buf = torch.zeros((B, L, H * d + 4), dtype=bf, device="cuda:0")
  buf[:, :, : H * d] = x.reshape(B, L, H * d)
  return buf[:, :, : H * d].unflatten(2, (H, d))


@pytest.mark.parametrize("L", [67, 258, 1002])
@pytest.mark.parametrize("d,with_mask,with_bias", [(64, True, True), (32, True, False), (128, False, True), (128, True, True)])
def test_weights_of_longer_rows_keep_their_bits(gpu, L, d, with_mask, with_bias):
  """Against 64 bits the matrix-core kernel is no further off than the general kernel, which multiplies 32-bit weights and which took
  these calls: both leave the output's rounding, sqrt(1/12) 2^-8 or so.  2 % is what the weights' second rounding, at 2^-17, and the
  order of the sums may add; weights rounded once to bf16 are 15 % and more further off."""
  rng = np.random.default_rng(L + d)
  B, H = 2, 2
  q, k, v = (O.round_bf16(rng.standard_normal((B, L, H, d)).astype(np.float32) * 0.4) for _ in range(3))
  mask = (rng.random((B, L, L)) > 0.3) & (np.arange(L)[None, None, :] <= np.arange(L)[None, :, None]) if with_mask else None
  bias = (rng.standard_normal((B, L, L)) * 0.4).astype(np.float32) if with_bias else None
  kw = dict(n=float(L), alpha=0.3, causal=not with_mask)
  want = O.hstu_attention_ref(q, k, v, mask=mask, bias=bias, dtype=np.float64, **kw)
  gk = dict(kw, mask=None if mask is None else _dev(mask), bias=None if bias is None else _dev(bias))
  ts = [_dev(x, bf) for x in (q, k, v)]
  err = lambda *t: np.linalg.norm(recml_amd.hstu_attention(*t, **gk).double().cpu().numpy() - want) / np.linalg.norm(want)
  here, general = err(*ts), err(*(_beside(t) for t in ts))
  assert here <= 1.02 * general, (here, general)


@pytest.mark.parametrize("d", [32, 128])
def test_a_mask_by_the_lowest_value(gpu, d):
  """A bias of finfo.min where a pair is not to count: weights of exactly 0, and gradients of 0, not NaN."""
  rng = np.random.default_rng(d)
  B, L, H = 2, 131, 2
  q, k, v, dout = (_dev(O.round_bf16(rng.standard_normal((B, L, H, d)).astype(np.float32) * 0.4), bf) for _ in range(4))
  mask = rng.random((B, L, L)) > 0.3
  low = _dev(np.where(mask, 0.0, np.finfo(np.float32).min).astype(np.float32)).requires_grad_(True)
  grads = []
  for bias, m in ((low, None), (torch.zeros_like(low).requires_grad_(True), _dev(mask))):
    ts = [t.clone().requires_grad_(True) for t in (q, k, v)]
    out = recml_amd.hstu_attention_autograd(*ts, n=float(L), causal=False, mask=m, bias=bias)
    grads.append([out.detach(), *torch.autograd.grad(out, [*ts, bias], dout)])
  for a, b in zip(*grads):
    assert a.isfinite().all() and (a.float() - b.float()).norm() <= 2.0 ** -8 * b.float().norm()


@pytest.mark.parametrize("keys", [16, 32, 48, 96, 144, 272])
@pytest.mark.parametrize("d,with_mask,with_bias", [(128, True, True), (128, True, False), (128, False, True), (64, True, True)])
def test_steps_of_the_dense_operands_ring(gpu, keys, d, with_mask, with_bias):
  """One to nine steps of 32 keys, odd and even, rows at both sides of a wave's 32; mask tiles that keep all, a part (a single pair dropped
  among them) and none, with other bytes than 1 for true.  Each of a row's activated weights and the output are rounded to bf16: 2^-8 of
  the largest."""
  rng = np.random.default_rng(keys + d)
  B, L, H = 2, 161, 2
  q = O.round_bf16(rng.standard_normal((B, L, H, d)).astype(np.float32) * 0.4)
  k, v = (O.round_bf16(rng.standard_normal((B, keys, H, d)).astype(np.float32) * 0.4) for _ in range(2))
  mask = np.ones((B, L, keys), np.uint8)
  mask[0, 5, keys - 1] = 0                       # one pair of an otherwise whole tile
  mask[0, 64:96, :16] = 0
  mask[1, 32:64] = 0                             # a wave's tiles
  mask[1, 128:] = rng.choice([0, 2, 255], (L - 128, keys))
  bias = (rng.standard_normal((B, L, keys)) * 0.4).astype(np.float32) if with_bias else None
  out = recml_amd.hstu_attention(_dev(q, bf), _dev(k, bf), _dev(v, bf), n=float(L), alpha=0.3, causal=False,
                                 mask=_dev(mask) if with_mask else None, bias=None if bias is None else _dev(bias))
  ref = O.pointwise_attention_dense(q * 0.3, k, v, (mask != 0).astype(np.float64) if with_mask else np.ones((B, L, keys)), bias)
  assert _rel(out.float().cpu().numpy(), ref) <= 2 * 2.0 ** -8
