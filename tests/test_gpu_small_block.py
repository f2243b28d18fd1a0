"""A whole block in one launch (short sequences, head dims of 16) against the same block in its steps, which a call that wants gradients
takes."""

import pytest
import torch

from recml_amd import _lib_block
from recml_amd.hstu_layer import HSTUBlock

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


def test_shapes_beside_it(gpu):
  assert not any([_taken(4, 65, 4), _taken(4, 50, 8), _taken(4, 50, 1), _taken(0, 50, 4), _taken(4, 0, 4), _taken(8192, 24, 4)])
  assert _taken(8192, 50, 4) == 1
