"""A block's calls in the forms that a user's program brings them in: the native call, the steps beside it and a training call agree on
what is computed, whatever the types and layouts of lengths, tables and parameters are."""

import numpy as np
import pytest
import torch
import torch.nn.utils.parametrize
import torch.nn.utils.prune

import recml_amd
from recml_amd import hstu_block_ops
from recml_amd.hstu_layer import HSTUBlock

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16
B, L, H, HD = 3, 96, 2, 64
D = H * HD


def _block(D=D, H=H, **kw):
  blk = HSTUBlock(D, H, dtype=BF, device=DEV, generator=torch.Generator().manual_seed(5), **kw)
  return blk


def _inputs(D=D):
  g = torch.Generator().manual_seed(2)
  x = (torch.randn((B, L, D), generator=g) * 0.5).to(DEV).to(BF)
  lens = torch.tensor([L, 41, 1], dtype=torch.int32, device=DEV)
  pos = (torch.randn((H, 2 * L - 1), generator=g) * 0.3).to(DEV)
  ts = torch.cumsum(torch.randint(1, 5000, (B, L), generator=g), 1).to(DEV)
  tsb = (torch.randn((H, 129), generator=g) * 0.3).to(DEV)
  return x, lens, pos, ts, tsb


def test_a_dense_mask_stands_alone(gpu):
  """Lengths and tables given beside a dense mask are not looked at, in inference as in training."""
  blk = _block()
  x, lens, pos, ts, tsb = _inputs()
  mask = torch.rand((B, L, L), generator=torch.Generator().manual_seed(3)).to(DEV) < 0.5
  more = dict(seq_lens=lens, pos_bias=pos, timestamps=ts, ts_bias=tsb)
  want = blk(x, attention_mask=mask)
  assert torch.equal(blk(x, attention_mask=mask, **more), want)
  blk.requires_grad_(True)
  trained = blk(x, attention_mask=mask, **more)
  # (bf16 on both sides, rounded at different steps: 2^-8 each)
  assert (trained.detach() - want).float().norm() <= 2e-2 * want.float().norm()


def _off_native(kind):
  """A block that the native call does not take, and its inputs' width."""
  if kind == "head dim 4":
    return _block(40, 10), 40
  blk = _block()
  if kind == "weights laid out across":
    blk.u_kernel.data = blk.u_kernel.data.permute(2, 1, 0).contiguous().permute(2, 1, 0)
  else:
    flat = torch.zeros(D + 1, dtype=BF, device=DEV)
    flat[1:] = 1.0
    blk.input_ln_gamma.data, blk.attn_ln_gamma.data = flat[1:], flat[1:].view(H, HD)
  return blk, D


@pytest.mark.parametrize("kind", ["head dim 4", "weights laid out across", "norm scales off a 16-byte boundary"])
@pytest.mark.parametrize("packed", [False, True])
def test_blocks_beside_the_native_call_keep_the_fused_steps(gpu, monkeypatch, kind, packed):
  """In bf16 the norm and the gate are one pass with one rounding, with and without gradients, also where the native call does not
  apply; against torch's steps, which round the normed rows by themselves (2^-8 apart per step)."""
  blk, width = _off_native(kind)
  x, lens, *_ = _inputs(width)
  valid = torch.arange(L, device=DEV)[None] < lens[:, None]
  offsets = torch.tensor(np.concatenate([[0], np.cumsum(lens.cpu().numpy())]), dtype=torch.int32, device=DEV)
  if packed:
    x = x[valid].contiguous()
  call = lambda t: blk.forward_jagged(t, offsets, L) if packed else blk(t, seq_lens=lens)
  norms, gates = [], []
  fwd, bwd = hstu_block_ops._norm_gate_fwd, hstu_block_ops.norm_gate_bwd
  monkeypatch.setattr(hstu_block_ops, "_norm_gate_fwd", lambda *a: norms.append(a[1] is not None) or fwd(*a))
  monkeypatch.setattr(hstu_block_ops, "norm_gate_bwd", lambda *a, **k: gates.append(a[1] is not None) or bwd(*a, **k))
  scored = call(x)
  assert norms == [False, True]                       # the input norm, then the attention norm with the gate
  blk.requires_grad_(True)
  dout = torch.randn(x.shape, generator=torch.Generator().manual_seed(9)).to(DEV).to(BF)
  wrt = [x.requires_grad_(True), *blk.parameters()]
  trained = call(x)
  got = torch.autograd.grad(trained, wrt, dout)
  assert norms == [False, True] * 2 and gates == [True, False]
  blk._fused_training = lambda *a: False
  plain = call(x)
  want = torch.autograd.grad(plain, wrt, dout)
  assert len(norms) == 4
  close = lambda a, b, tol: (a.float() - b.float()).norm() <= tol * b.float().norm()
  assert close(scored, plain.detach(), 1e-2) and close(trained.detach(), plain.detach(), 1e-2)
  for g, w, name in zip(got, want, ["x", *dict(blk.named_parameters())]):
    assert close(g, w, 3e-2), name


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("grad", [False, True])
def test_other_integer_and_table_types_take_the_native_call(gpu, monkeypatch, packed, grad):
  """torch's default integers for lengths and offsets, 32-bit timestamps, a bf16 table, one whose rows are strided: the same bits as with
  the kernels' own types, through the native call, and table gradients in the tables' own types."""
  blk = _block().requires_grad_(grad)
  x, lens, pos, ts, tsb = _inputs()
  pos16 = pos.to(BF)
  wide = torch.zeros((H, 2 * 129), device=DEV)
  wide[:, ::2] = tsb
  ts = ts - ts.min()
  offsets = torch.tensor(np.concatenate([[0], np.cumsum(lens.cpu().numpy())]), dtype=torch.int32, device=DEV)
  if packed:
    valid = torch.arange(L, device=DEV)[None] < lens[:, None]
    x, ts = x[valid].contiguous(), ts[valid].contiguous()
  call = lambda lens, offsets, **kw: blk.forward_jagged(x, offsets, L, **kw) if packed else blk(x, seq_lens=lens, **kw)
  seen = []
  native = recml_amd._native.block
  monkeypatch.setattr(recml_amd._native, "block", lambda *a: (seen.append(native(*a)), seen[-1])[1])
  plain = [t.requires_grad_(grad) for t in (pos16.float(), tsb.clone())]
  given = [t.requires_grad_(grad) for t in (pos16, wide[:, ::2])]
  want = call(lens, offsets, pos_bias=plain[0], timestamps=ts, ts_bias=plain[1])
  got = call(lens.long(), offsets.long(), pos_bias=given[0], timestamps=ts.int(), ts_bias=given[1])
  assert len([s for s in seen if s is not None]) == 2
  assert torch.equal(got, want)
  if grad:
    dout = torch.randn(x.shape, generator=torch.Generator().manual_seed(9)).to(DEV).to(BF)
    params = list(blk.parameters())
    a, b = torch.autograd.grad(got, [*given, *params], dout), torch.autograd.grad(want, [*plain, *params], dout)
    assert a[0].dtype == BF
    # (the tables' sums are added to by atomics, in no fixed order)
    assert (a[0].float() - b[0]).abs().max() <= 2.0 ** -8 * b[0].abs().max() and (a[1] - b[1]).abs().max() <= 1e-5 * b[1].abs().max()
    assert all(torch.equal(p, q) for p, q in zip(a[2:], b[2:]))


def test_converted_lengths_are_shared_and_not_outlived(gpu, monkeypatch):
  """The blocks of a model share one preparation from 64-bit lengths too, and lengths changed in place are seen."""
  from recml_amd import hstu_ops
  made = []

  class Batch(hstu_ops.AttentionBatch):
    def __init__(self):
      super().__init__()
      made.append(self)

  monkeypatch.setattr(hstu_ops, "AttentionBatch", Batch)
  model = recml_amd.HSTU(vocab_size=50, max_positions=L, model_dim=D, num_heads=H, num_layers=3, dtype=BF, device=DEV, add_head=False, seed=1)
  ids = torch.randint(1, 50, (B, L), generator=torch.Generator().manual_seed(4)).to(DEV)
  lens, pos = _inputs()[1:3]
  assert torch.equal(model(ids, seq_lens=lens.long(), pos_bias=pos), model(ids, seq_lens=lens, pos_bias=pos))
  assert [b.prepared_calls for b in made] == [2, 2]
  blk, batch, wide = _block(), hstu_ops.AttentionBatch(), lens.long()
  x = _inputs()[0]
  blk(x, seq_lens=wide, pos_bias=pos, batch=batch)
  wide.fill_(30)
  assert torch.equal(blk(x, seq_lens=wide, pos_bias=pos, batch=batch), blk(x, seq_lens=torch.full_like(lens, 30), pos_bias=pos))


class _Doubled(torch.nn.Module):
  def forward(self, w):
    return 2.0 * w


@pytest.mark.parametrize("how", ["parametrize", "prune", "prune a bias"])
@pytest.mark.parametrize("packed", [False, True])
def test_parametrized_and_pruned_blocks(gpu, how, packed):
  """torch.nn.utils.parametrize and prune take a parameter's name out of the module's parameters and put a tensor there: the same as a
  block with that tensor, and the gradient reaches the parameter behind it."""
  x, lens, *_ = _inputs()
  offsets = torch.tensor([0, L, L + 41, L + 42], dtype=torch.int32, device=DEV)
  call = lambda blk: blk.forward_jagged(x[:, 0].repeat(50, 1)[: L + 42].contiguous(), offsets, L) if packed else blk(x, seq_lens=lens)
  blk, plain = _block(use_bias=True), _block(use_bias=True)
  for b in (blk, plain):
    b.requires_grad_(True)
    b.q_bias.data += 0.25
  if how == "parametrize":
    torch.nn.utils.parametrize.register_parametrization(blk, "u_kernel", _Doubled(), unsafe=True)
    behind, shown = blk.parametrizations.u_kernel.original, plain.u_kernel
    shown.data *= 2.0
    factor = torch.full_like(shown, 2.0)
  else:
    name = "output_kernel" if how == "prune" else "q_bias"
    factor = (torch.rand(getattr(blk, name).shape, generator=torch.Generator().manual_seed(1)) < 0.5).to(DEV).to(BF)
    torch.nn.utils.prune.custom_from_mask(blk, name, factor)
    behind, shown = getattr(blk, name + "_orig"), getattr(plain, name)
    shown.data *= factor
  got, want = call(blk), call(plain)
  assert torch.equal(got, want)
  dout = torch.randn(got.shape, generator=torch.Generator().manual_seed(9)).to(DEV).to(BF)
  a, b = torch.autograd.grad(got, behind, dout)[0], torch.autograd.grad(want, shown, dout)[0]
  assert torch.equal(a, b * factor)
  with torch.no_grad():
    assert torch.equal(call(blk), call(plain))
