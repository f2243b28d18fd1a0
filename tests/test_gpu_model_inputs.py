"""The model's front end in training: what its gradients depend on, and what it does with ids and lengths out of range."""

import pytest
import torch

import recml_amd

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16
B, L, D, V = 3, 40, 64, 60


def _model(**kw):
  model = recml_amd.HSTU(vocab_size=V, max_positions=L, model_dim=D, num_heads=2, num_layers=1, add_head=False, dtype=BF, device=DEV, seed=3, **kw)
  return model.requires_grad_(True)


def _inputs():
  g = torch.Generator().manual_seed(1)
  ids = torch.randint(1, V, (B, L), generator=g).to(DEV)
  lens = torch.tensor([L, 17, 1], dtype=torch.int32, device=DEV)
  return ids, lens, torch.randn((B, L, D), generator=g).to(DEV).to(BF)


def _grads(model, out, dout):
  return dict(zip([n for n, _ in model.named_parameters()], torch.autograd.grad(out, list(model.parameters()), dout)))


@pytest.mark.parametrize("jagged", [False, True])
@pytest.mark.parametrize("change", ["ids", "table through .data", "table in place", "position table in place"])
def test_gradients_do_not_depend_on_what_becomes_of_the_inputs(gpu, jagged, change):
  """A training loop that refills its id buffer, or updates a table, between forward and backward: the same bits as without."""
  model = _model(scale_by_sqrt_dim=True)
  ids, lens, dout = _inputs()
  want = _grads(model, model(ids, seq_lens=lens, jagged=jagged), dout)
  out = model(ids, seq_lens=lens, jagged=jagged)
  with torch.no_grad():
    if change == "ids":
      ids.fill_(2)
    elif change == "table through .data":
      model.item_embedding.data.add_(1.0)
    else:
      (model.item_embedding if change == "table in place" else model.position_embedding).add_(1.0)
  got = _grads(model, out, dout)
  for name in want:
    assert torch.equal(got[name], want[name]), name
