"""What torch's own machinery expects of the native calls: error types, forward-mode gradients, saved-tensor hooks, frozen parts."""

import pytest
import torch

import recml_amd
from recml_amd.hstu_layer import HSTUBlock

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


def _randn(*shape, seed=0, std=0.5, dtype=BF):
  return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * std).to(DEV).to(dtype)


def _block(D=128, H=2, **kw):
  return HSTUBlock(D, H, dtype=BF, device=DEV, generator=torch.Generator().manual_seed(5), **kw)


@pytest.mark.parametrize("grad", [False, True])
def test_out_of_memory_keeps_its_type(gpu, grad):
  """torch.OutOfMemoryError is what programs catch to try again with less."""
  q = torch.zeros((1, 1, 2, 128), dtype=BF, device=DEV, requires_grad=grad).expand(1, 1 << 22, 2, 128)      # (a result of 2 GB)
  op = recml_amd.hstu_attention_autograd if grad else recml_amd.hstu_attention
  blk = _block().requires_grad_(grad)
  x = torch.zeros((1, 1 << 19, 128), dtype=BF, device=DEV)                                                  # (a projection of 512 MB)
  lens = torch.tensor([5], dtype=torch.int32, device=DEV)
  torch.cuda.synchronize()
  torch.cuda.empty_cache()
  torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / torch.cuda.get_device_properties(0).total_memory)
  try:
    with pytest.raises(torch.OutOfMemoryError):
      op(q, q, q, seq_lens=lens)
    with pytest.raises(torch.OutOfMemoryError):
      blk(x, seq_lens=lens)
  finally:
    torch.cuda.set_per_process_memory_fraction(1.0)


@pytest.mark.parametrize("grad", [False, True])
def test_forward_mode_is_refused_not_dropped(gpu, grad):
  """The kernels give no tangents: a dual tensor anywhere in a differentiable call is refused, as torch's autograd functions refuse it."""
  lens = torch.tensor([40, 7], dtype=torch.int32, device=DEV)
  q = _randn(2, 40, 2, 64)
  pos = _randn(2, 79, std=0.1, dtype=torch.float32)
  blk = _block().requires_grad_(grad)
  x = _randn(2, 40, 128)
  gamma, beta = torch.ones(128, dtype=BF, device=DEV), torch.zeros(128, dtype=BF, device=DEV)
  model = recml_amd.HSTU(vocab_size=50, max_positions=40, model_dim=128, num_heads=2, num_layers=1, dtype=BF, device=DEV, seed=1, add_head=False)
  model.requires_grad_(grad)
  ids = torch.randint(1, 50, (2, 40), generator=torch.Generator().manual_seed(4)).to(DEV)
  with torch.autograd.forward_ad.dual_level():
    dual = lambda t: torch.autograd.forward_ad.make_dual(t.detach(), torch.ones_like(t))
    calls = [lambda: recml_amd.hstu_attention_autograd(dual(q), q, q, seq_lens=lens),
             lambda: recml_amd.hstu_attention_autograd(q, q, q, seq_lens=lens, pos_bias=dual(pos)),
             lambda: blk(dual(x), seq_lens=lens), lambda: blk(x, seq_lens=lens, pos_bias=dual(pos)),
             lambda: blk.forward_jagged(dual(x[0]), torch.tensor([0, 40], dtype=torch.int32, device=DEV), 40),
             lambda: recml_amd.layer_norm(dual(x), gamma, beta), lambda: recml_amd.norm_gate(x, x, dual(gamma), beta),
             lambda: model(ids, seq_lens=lens, pos_bias=dual(pos[0]))]
    for i, call in enumerate(calls):
      with pytest.raises(NotImplementedError):
        call()
        pytest.fail(f"call {i} took a dual tensor")


def test_the_head_carries_tangents_and_second_derivatives(gpu):
  """The output head stands for x @ w, which has both.  bf16 products of 64 and 96 terms, rounded once on either side: 2^-8."""
  model = recml_amd.HSTU(vocab_size=96, max_positions=8, model_dim=64, num_heads=1, num_layers=0, dtype=BF, device=DEV, seed=1)
  model.requires_grad_(True)
  x, t, v, u = _randn(3, 8, 64, seed=1).requires_grad_(True), _randn(3, 8, 64, seed=2), _randn(3, 8, 96, seed=3), _randn(3, 8, 64, seed=4)
  w = model.reverse_embedding
  close = lambda a, b: (a.float() - b.float()).norm() <= 2.0 ** -8 * b.float().norm()
  with torch.autograd.forward_ad.dual_level():
    tangent = torch.autograd.forward_ad.unpack_dual(model._head(torch.autograd.forward_ad.make_dual(x.detach(), t))).tangent
    assert tangent is not None and close(tangent, t.float() @ w.detach().float())
  y = model._head(x)
  gx, gw = torch.autograd.grad(y, [x, w], v, create_graph=True)
  assert close(gx, v.float() @ w.detach().float().t())
  got = torch.autograd.grad([gx, gw], [w, x], [u, torch.ones_like(gw)])
  assert close(got[0], u.reshape(-1, 64).float().t() @ v.reshape(-1, 96).float())
  assert close(got[1], v.float() @ torch.ones(96, 64, device=DEV))


def _bytes(t):
  return t.numel() * t.element_size()


@pytest.mark.parametrize("packed", [False, True])
def test_saved_tensor_hooks_see_what_the_block_keeps(gpu, packed):
  """The block's intermediates (the normed rows, the projection before and after its activation, the attention and the gated rows: 11 x
  tokens x D) go through torch's saved-tensor hooks: save_on_cpu leaves none of them on the GPU, and the gradients are the same bits."""
  T, D = 4096, 128
  blk = _block().requires_grad_(True)
  x = _randn(T, D).requires_grad_(True)
  offsets = torch.arange(0, T + 1, 512, dtype=torch.int32, device=DEV)
  call = lambda: blk.forward_jagged(x, offsets, 512) if packed else blk(x.view(8, 512, D), seq_lens=torch.full((8,), 512, dtype=torch.int32, device=DEV))
  dout = _randn(*call().shape, seed=3)
  want = torch.autograd.grad(call(), [x, *blk.parameters()], dout)
  held = []
  for hooks in (None, torch.autograd.graph.save_on_cpu()):
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    if hooks is None:
      out = call()
    else:
      with hooks:
        out = call()
    held.append(torch.cuda.memory_allocated() - before)
    got = torch.autograd.grad(out, [x, *blk.parameters()], dout)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    del out, got
  assert held[0] >= 11 * _bytes(x) and held[1] <= 2 * _bytes(x)


def test_checkpointing_a_block_frees_and_recomputes(gpu):
  """torch.utils.checkpoint without reentry replaces what is saved: nothing but the output stays, and the gradients are the same bits,
  dropout included (its seed comes from torch's generator, which checkpointing restores)."""
  from torch.utils.checkpoint import checkpoint
  T, D = 4096, 128
  blk = _block(dropout=0.2).requires_grad_(True)
  x = _randn(8, 512, D).requires_grad_(True)
  lens = torch.full((8,), 500, dtype=torch.int32, device=DEV)
  dout = _randn(8, 512, D, seed=3)
  torch.manual_seed(11)
  want = torch.autograd.grad(blk(x, seq_lens=lens), [x, *blk.parameters()], dout)
  torch.manual_seed(11)
  torch.cuda.synchronize()
  before = torch.cuda.memory_allocated()
  out = checkpoint(lambda t: blk(t, seq_lens=lens), x, use_reentrant=False)
  assert torch.cuda.memory_allocated() - before <= 2 * _bytes(x)
  got = torch.autograd.grad(out, [x, *blk.parameters()], dout)
  assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_a_second_backward_needs_the_graph_kept(gpu):
  blk = _block().requires_grad_(True)
  x = _randn(2, 40, 128).requires_grad_(True)
  out = blk(x, seq_lens=torch.tensor([40, 9], dtype=torch.int32, device=DEV))
  dout = _randn(2, 40, 128, seed=1)
  a = torch.autograd.grad(out, x, dout, retain_graph=True)[0]
  assert torch.equal(torch.autograd.grad(out, x, dout)[0], a)
  with pytest.raises(RuntimeError, match="second time"):
    torch.autograd.grad(out, x, dout)


@pytest.mark.parametrize("part", ["output_kernel", "output_bias", "attn_ln_beta", "pos", "k_kernel", "v_bias", "input_ln_gamma", "x"])
def test_frozen_parts_are_not_differentiated(gpu, part):
  """A gradient is taken back only as far as something behind wants it, and only what that reads is kept: the same bits as with
  everything trained, and for the parts behind the gate neither the projection nor its gradient (8 x tokens x D) is there."""
  T, D = 4096, 128
  blk = _block(use_bias=True)
  x = _randn(8, 512, D)
  lens = torch.full((8,), 500, dtype=torch.int32, device=DEV)
  pos = _randn(2, 1023, std=0.1, dtype=torch.float32)
  dout = _randn(8, 512, D, seed=3)
  named = dict(blk.named_parameters(), x=x, pos=pos)
  for t in named.values():
    t.requires_grad_(True)
  want = dict(zip(named, torch.autograd.grad(blk(x, seq_lens=lens, pos_bias=pos), list(named.values()), dout)))[part]
  for t in named.values():
    t.requires_grad_(False)
  named[part].requires_grad_(True)
  torch.cuda.synchronize()
  before = torch.cuda.memory_allocated()
  out = blk(x, seq_lens=lens, pos_bias=pos)
  held = torch.cuda.memory_allocated() - before
  torch.cuda.reset_peak_memory_stats()
  got = torch.autograd.grad(out, named[part], dout)[0]
  peak = torch.cuda.max_memory_allocated() - before
  # (the position table's gradient is added up by atomics, in no fixed order)
  assert torch.equal(got, want) if part != "pos" else (got - want).abs().max() <= 1e-5 * want.abs().max()
  if part.startswith("output"):
    # (a bias's column sum is torch's, which brings 4 MB of scratch, 4 x tokens x D here)
    assert held <= 3 * _bytes(x) and peak <= 7 * _bytes(x)
