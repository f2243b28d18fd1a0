"""A whole block in one launch (short sequences, head dims of 16) against the same block in its steps, which a call that wants gradients
takes."""

import numpy as np
import pytest
import torch

from oracle import hstu_block_oracle as BO
from recml_amd import _lib_block, hstu_layer
from recml_amd.hstu_layer import HSTU, HSTUBlock

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


def _taken(B, L, H):
  return _lib_block.load().hstu_block_small_takes(B, L, H, 16, 16 * H)


@pytest.mark.parametrize("B,L,H,lens,pos,biases,jagged", [
    (1, 1, 2, [1], None, False, False),
    (3, 16, 4, [16, 0, 1], None, True, False),           # a whole block of queries, an empty sequence
    (3, 17, 2, [17, 16, 3], "shared", False, False),     # one row past it
    (2, 33, 4, [33, 32], "heads", True, False),          # one past a block of the products
    (2, 64, 4, [64, 63], None, False, False),            # every row
    (4, 50, 4, [50, 7, 50, 33], "heads", False, True),
    (3, 64, 2, [1, 64, 0], "shared", True, True),        # packed, an empty sequence at the end
])
def test_block_in_one_launch(gpu, B, L, H, lens, pos, biases, jagged):
  assert _taken(B, L, H) == 1
  D = 16 * H
  g = torch.Generator().manual_seed(B * L)
  blk = HSTUBlock(D, H, dtype=BF, device=DEV, use_bias=biases, generator=g)
  with torch.no_grad():
    for prm in blk.parameters():
      prm.add_((torch.randn(prm.shape, generator=g) * 0.1).to(DEV).to(BF))
  x = torch.randn((B, L, D), generator=g).to(DEV).to(BF)
  lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
  tab = None if pos is None else (torch.randn((H if pos == "heads" else 1, 2 * L - 1), generator=g) * 0.3).to(DEV)

  def run(t):
    if not jagged:
      return blk(t, seq_lens=lens, pos_bias=tab)
    keep = torch.arange(L, device=DEV)[None] < lens[:, None]
    offsets = torch.cat([lens.new_zeros(1), lens.cumsum(0).to(torch.int32)])
    return blk.forward_jagged(t[keep].contiguous(), offsets, L, pos_bias=tab)

  with torch.no_grad():
    got = run(x)
  blk.requires_grad_(True)
  want = run(x).detach()
  assert got.shape == want.shape
  # The form with gradients rounds u, q, k and v once more, ahead of their activation (2^-9 of each), and sums in another order flip
  # roundings of the steps behind.  u, and q, k, v through the weights and their sums, each move the block's branch by 2^-9 at most on
  # average: 2^-7 for the four together, and twice that in single values.
  diff = (got.float() - want.float()).abs()
  assert diff.max() <= 2.0 ** -6 * want.float().abs().max()
  assert diff.norm() <= 2.0 ** -7 * want.float().norm()
  if not jagged:
    # what stands in the padding is nobody's business
    bad = torch.where((torch.arange(L, device=DEV)[None] < lens[:, None])[..., None], x, torch.full_like(x, float("nan")))
    with torch.no_grad():
      got_bad = run(bad)
    for b in range(B):
      assert torch.equal(got_bad[b, :lens[b]], got[b, :lens[b]])


@pytest.mark.parametrize("B,L,H,lens,pos,biases", [
    (1, 1, 2, [1], None, False),
    (3, 17, 2, [17, 16, 3], "shared", True),
    (2, 33, 4, [33, 32], "heads", True),
    (2, 64, 4, [64, 63], None, False),
    (4, 50, 4, [50, 7, 50, 33], "heads", False),
])
def test_against_the_oracle(gpu, B, L, H, lens, pos, biases):
  """The launch against the block in 64 bits.  Five of its values are rounded to 8 bits, one behind the other (normed; u, q, k, v; the
  attention; gated; the output): 2^-9 / sqrt(3) each in the mean, with signs that do not agree, so sqrt(5) of that for the rows' norm:
  2^-8.6; single values up to four times as far."""
  assert _taken(B, L, H) == 1
  D = 16 * H
  g = torch.Generator().manual_seed(7 * B + L)
  blk = HSTUBlock(D, H, dtype=BF, device=DEV, use_bias=biases, generator=g)
  with torch.no_grad():
    for prm in blk.parameters():
      prm.add_((torch.randn(prm.shape, generator=g) * 0.1).to(DEV).to(BF))
  x = torch.randn((B, L, D), generator=g).to(BF)
  tab = None if pos is None else torch.randn((H if pos == "heads" else 1, 2 * L - 1), generator=g) * 0.3
  with torch.no_grad():
    got = blk(x.to(DEV), seq_lens=torch.tensor(lens, dtype=torch.int32, device=DEV), pos_bias=None if tab is None else tab.to(DEV))
  got = got.double().cpu().numpy()
  w = {k: v.detach().double().cpu().numpy() for k, v in blk.named_parameters()}
  for b in range(B):
    n = lens[b]
    want = _oracle(x[b, :n].double().numpy(), w, H, L, tab)
    diff = np.abs(got[b, :n] - want)
    assert np.linalg.norm(diff) <= 2.0 ** -8 * np.linalg.norm(want)
    assert diff.max() <= 2.0 ** -7 * np.abs(want).max()


def _oracle(x, w, H, L, tab):
  """What BO.hstu_block does for one sequence in a batch of length L, with a table per head (BO.hstu_block has one for all heads)."""
  n, D = x.shape
  hd = D // H
  f = lambda name: w[name].reshape((D, H, hd) if name.endswith("_kernel") and name[0] in "uqkv" else (H, hd, D) if name == "output_kernel" else
                                   (H, hd) if name.startswith("attn_ln") or (name.endswith("_bias") and name[0] in "uqkv") else (D,))
  normed = BO.layer_norm(x, f("input_ln_gamma"), f("input_ln_beta"), 1e-6)
  proj = {}
  for c in "uqkv":
    y = np.einsum("td,dnh->tnh", normed, f(c + "_kernel"))
    proj[c] = BO.O.silu(y + f(c + "_bias") if c + "_bias" in w else y)
  s = np.einsum("inh,jnh->nij", proj["q"], proj["k"])
  if tab is not None:
    i = np.arange(n)
    s = s + tab.double().numpy()[:, (L - 1) + i[None, :] - i[:, None]]
  p = np.where(np.tril(np.ones((n, n), bool))[None], BO.O.silu(s), 0.0) / L
  attn = BO.layer_norm(np.einsum("nij,jnh->inh", p, proj["v"]), f("attn_ln_gamma"), f("attn_ln_beta"), 1e-6, axes=(-2, -1))
  out = np.einsum("tnh,nhd->td", proj["u"] * attn, f("output_kernel")) + x
  return out + f("output_bias") if "output_bias" in w else out


def test_shapes_beside_it(gpu):
  assert not any([_taken(4, 65, 4), _taken(4, 50, 8), _taken(4, 50, 1), _taken(0, 50, 4), _taken(4, 0, 4), _taken(8192, 24, 4)])
  assert _taken(8192, 50, 4) == 1


def _model(layers, D, H, L, biases=False, seed=0):
  g = torch.Generator().manual_seed(seed)
  model = HSTU(vocab_size=300, max_positions=L, model_dim=D, num_heads=H, num_layers=layers, add_head=False, dtype=BF, device=DEV, seed=seed)
  if biases:
    model.decoder_blocks = torch.nn.ModuleList(HSTUBlock(D, H, dtype=BF, device=DEV, use_bias=True, generator=g) for _ in range(layers))
  with torch.no_grad():
    for prm in model.parameters():
      prm.add_((torch.randn(prm.shape, generator=g) * 0.05).to(DEV).to(BF))
  return model, g


@pytest.mark.parametrize("layers,B,L,H,pos,biases,jagged", [
    (1, 3, 17, 4, None, True, False),
    (2, 2, 64, 2, "heads", False, False),
    (4, 5, 50, 4, "shared", True, True),
    (17, 2, 33, 4, "heads", False, False),               # one block more than a launch takes
    (33, 3, 20, 2, None, False, True),                   # three launches
])
def test_blocks_in_one_launch_are_the_blocks_one_by_one(gpu, layers, B, L, H, pos, biases, jagged):
  """The same bits as one launch a block, which a hook on a block (or a subclass's forward) brings back."""
  D = 16 * H
  model, g = _model(layers, D, H, L, biases, seed=layers)
  ids = torch.randint(1, 300, (B, L), generator=g).to(DEV)
  lens = torch.randint(1, L + 1, (B,), generator=g).int()
  lens[0] = L
  tab = None if pos is None else (torch.randn((H if pos == "heads" else 1, 2 * L - 1), generator=g) * 0.3).to(DEV)
  calls, own = [], hstu_layer._native.block
  with torch.no_grad(), pytest.MonkeyPatch.context() as patch:
    patch.setattr(hstu_layer._native, "block", lambda *a: calls.append(1) or own(*a))
    got = model(ids, seq_lens=lens.to(DEV), pos_bias=tab, jagged=jagged)
    assert not calls
    seen = []
    if jagged:
      patch.setattr(HSTUBlock, "forward_jagged", lambda self, *a, f=HSTUBlock.forward_jagged, **kw: seen.append(1) or f(self, *a, **kw))
    else:
      for blk in model.decoder_blocks:
        blk.register_forward_hook(lambda *a: seen.append(1) and None)
    want = model(ids, seq_lens=lens.to(DEV), pos_bias=tab, jagged=jagged)
    assert len(seen) == layers and len(calls) == layers
  # the closing norm's sums are in another order (one place of its bf16 rows); the packed form's closing norm is the same kernel
  if jagged:
    assert torch.equal(got, want)
  else:
    assert bool(((got.float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs() + 2.0 ** -20).all())


def test_what_keeps_the_blocks_apart(gpu):
  """Gradients, other sizes among the blocks, dropout in training, a global hook: each block is called by itself."""
  model, g = _model(2, 32, 2, 20)
  ids = torch.randint(1, 300, (2, 20), generator=g).to(DEV)
  kw = dict(seq_lens=torch.tensor([20, 5], dtype=torch.int32, device=DEV))
  calls, own = [], hstu_layer._native.block
  with pytest.MonkeyPatch.context() as patch:
    patch.setattr(hstu_layer._native, "block", lambda *a: calls.append(1) or own(*a))

    def count(f):
      calls.clear()
      f()
      return len(calls)

    run = lambda: model(ids, **kw)
    assert count(run) == 0
    handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert count(run) == 2
    handle.remove()
    model.decoder_blocks[1].eps = 1e-3
    assert count(run) == 2
    model.decoder_blocks[1].eps = model.decoder_blocks[0].eps
    model.decoder_blocks[1].dropout = 0.5
    assert count(run) == 2 and count(lambda: model.eval()(ids, **kw)) == 0
    model.requires_grad_(True)
    assert count(run) == 2
    with torch.no_grad():
      assert count(run) == 0
