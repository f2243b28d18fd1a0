"""A block's calls in the forms that a user's program brings them in: the native call, the steps beside it and a training call agree on
what is computed, whatever the types and layouts of lengths, tables and parameters are."""

import numpy as np
import pytest
import torch

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
