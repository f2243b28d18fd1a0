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


@pytest.fixture
def little_memory(gpu):
  torch.cuda.synchronize()
  torch.cuda.empty_cache()
  total = torch.cuda.get_device_properties(0).total_memory
  torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)
  yield
  torch.cuda.set_per_process_memory_fraction(1.0)


@pytest.mark.parametrize("grad", [False, True])
def test_out_of_memory_keeps_its_type(little_memory, grad):
  """torch.OutOfMemoryError is what programs catch to try again with less."""
  q = torch.zeros((1, 1, 2, 128), dtype=BF, device=DEV, requires_grad=grad).expand(1, 1 << 17, 2, 128)
  op = recml_amd.hstu_attention_autograd if grad else recml_amd.hstu_attention
  with pytest.raises(torch.OutOfMemoryError):
    op(q, q, q, seq_lens=torch.tensor([5], dtype=torch.int32, device=DEV))
  blk = _block().requires_grad_(grad)
  x = torch.zeros((1, 1 << 16, 128), dtype=BF, device=DEV)
  with pytest.raises(torch.OutOfMemoryError):
    blk(x, seq_lens=torch.tensor([5], dtype=torch.int32, device=DEV))
