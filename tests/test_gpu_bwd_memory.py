"""The scratch of a backward pass: what it asks for, and what it does where the device has not that much."""

import pytest
import torch

import recml_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wanted", [True, False])
def test_a_block_asks_for_what_its_attention_takes(gpu, wanted):
  """Heads of 64 with a position table: whether dS is handed on goes by whether the table's gradient is wanted, so a block asks once all of
  its call is filled in."""
  B, L, H, d = 4, 4096, 4, 64
  torch.manual_seed(0)
  layer = recml_amd.HSTUBlock(H * d, H).cuda().to(torch.bfloat16)
  x = torch.randn(B, L, H * d, device="cuda").mul_(0.5).to(torch.bfloat16).requires_grad_()
  pos = (torch.randn(H, 2 * L - 1, device="cuda") * 0.1).requires_grad_(wanted)
  out = layer(x, pos_bias=pos)
  assert out.grad_fn.name() == "HstuBlockBackward"
  kept = B * H * L * L            # (two bytes for each of half the pairs)
  torch.cuda.synchronize()
  torch.cuda.reset_peak_memory_stats()
  before = torch.cuda.memory_allocated()
  torch.autograd.grad(out, [x, pos] if wanted else [x], torch.randn_like(out))
  assert (torch.cuda.max_memory_allocated() - before > kept) == wanted
