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


@pytest.mark.parametrize("rows", [32, 192])
def test_position_gradient_of_a_padded_batch_is_one_sum(gpu, rows):
  """The position table is broadcast over a padded batch: its gradient against the front end in float64.  Each row's gradient is rounded
  to bf16 (2^-9 of it at most, independently) and the sum over the batch once more: 2^-8 in all; rounded at every addition it would be
  7e-3 off for 32 sequences and 1.7e-2 for 192."""
  g = torch.Generator().manual_seed(rows)
  model = recml_amd.HSTU(vocab_size=500, max_positions=8, model_dim=128, num_heads=2, num_layers=0, add_head=False, dtype=BF, device=DEV, seed=3)
  model.requires_grad_(True)
  ids = torch.randint(0, 500, (rows, 8), generator=g).to(DEV)
  dout = torch.randn((rows, 8, 128), generator=g).to(DEV).to(BF)
  # (one norm alone: the model's closing norm on top of it would hide the front end's rounding behind its own)
  x = model._front_end(ids)[0]
  got = torch.autograd.grad(x, model.position_embedding, dout)[0].double()
  table, pos = model.item_embedding.detach().double(), model.position_embedding.detach().double().requires_grad_(True)
  summed = table[ids] + pos
  summed = summed + (summed.to(BF).double() - summed).detach()
  out = torch.nn.functional.layer_norm(summed, (128,), eps=1e-6)
  want = torch.autograd.grad(out, pos, dout.double())[0]
  assert (got - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("count", [2, 5])
@pytest.mark.parametrize("grad", [False, True])
def test_lengths_of_another_batch_size_are_refused(gpu, count, grad):
  """Packing is by the lengths: more of them than there are sequences would have the gather read past the ids."""
  model = _model()
  with torch.set_grad_enabled(grad), pytest.raises(RuntimeError):
    model(_inputs()[0], seq_lens=torch.full((count,), 7, dtype=torch.int32, device=DEV), jagged=True)


@pytest.mark.parametrize("jagged", [False, True])
def test_ids_out_of_the_vocabulary(gpu, jagged):
  """With gradients ids are taken as torch's indexing takes them: negative ones count from the end, others are an error.  Without,
  they are clamped."""
  model = _model()
  ids, lens, dout = _inputs()
  last, negative = ids.clone(), ids.clone()
  last[0, 3], negative[0, 3] = V - 1, -1
  want = _grads(model, model(last, seq_lens=lens, jagged=jagged), dout)
  got = _grads(model, model(negative, seq_lens=lens, jagged=jagged), dout)
  assert all(torch.equal(got[n], want[n]) for n in want)
  for bad in (V, -V - 1):
    out_of_range = ids.clone()
    out_of_range[0, 3] = bad
    with pytest.raises(IndexError):
      model(out_of_range, seq_lens=lens, jagged=jagged)
    with torch.no_grad():
      clamped = model(out_of_range.clamp(0, V - 1), seq_lens=lens, jagged=jagged)
      assert torch.equal(model(out_of_range, seq_lens=lens, jagged=jagged), clamped)
  # past the sequences' ends packed ids are never read
  out_of_range = ids.clone()
  out_of_range[2, 5] = V
  if jagged:
    assert model(out_of_range, seq_lens=lens, jagged=True).isfinite().all()


def test_positions_past_the_table(gpu):
  """A batch longer than the position table: an error with gradients, in the packed form where a token reaches past it."""
  model = _model()
  g = torch.Generator().manual_seed(1)
  ids = torch.randint(1, V, (B, L + 8), generator=g).to(DEV)
  lens = lambda n: torch.tensor([n, 17, 1], dtype=torch.int32, device=DEV)
  with pytest.raises(RuntimeError):
    model(ids, seq_lens=lens(L))
  assert model(ids, seq_lens=lens(L), jagged=True).isfinite().all()
  with pytest.raises(IndexError):
    model(ids, seq_lens=lens(L + 1), jagged=True)


@pytest.mark.parametrize("dropout", [0.0, 0.2])
@pytest.mark.parametrize("jagged", [False, True])
def test_a_mask_that_is_not_end_padded_ends_the_call(gpu, jagged, dropout):
  """The error comes before the work: no more than the first block is run, and nothing random is drawn."""
  model = recml_amd.HSTU(vocab_size=V, max_positions=L, model_dim=D, num_heads=2, num_layers=3, add_head=False, dtype=BF, device=DEV, dropout=dropout)
  ran = []
  for block in model.decoder_blocks:
    forward = block.forward, block.forward_jagged
    block.forward = lambda *a, f=forward[0], **k: ran.append(1) or f(*a, **k)
    block.forward_jagged = lambda *a, f=forward[1], **k: ran.append(1) or f(*a, **k)
  ids, lens, _ = _inputs()
  mask = torch.arange(L, device=DEV)[None] < lens[:, None]
  torch.manual_seed(3)
  before = torch.get_rng_state(), torch.cuda.get_rng_state()
  mask[1, 5] = False
  with pytest.raises(ValueError, match="end-padded"):
    model(ids, padding_mask=mask, jagged=jagged)
  assert len(ran) <= (0 if jagged or dropout else 1)
  assert torch.equal(torch.get_rng_state(), before[0]) and torch.equal(torch.cuda.get_rng_state(), before[1])
  mask[1, 5] = True
  assert model(ids, padding_mask=mask, jagged=jagged).isfinite().all()


@pytest.mark.parametrize("batch,length", [(1, 1), (3, 40), (5, 65), (9, 130)])
@pytest.mark.parametrize("grad", [False, True])
def test_lengths_from_the_mask_in_the_front_end(gpu, batch, length, grad):
  """A padding mask's lengths come with the front end's launch (four rows of it to a workgroup, 64 bytes to a wavefront): the same bits as
  the lengths themselves give, and a row that is not end-padded is refused, wherever it stands."""
  g = torch.Generator().manual_seed(length)
  model = recml_amd.HSTU(vocab_size=V, max_positions=length, model_dim=D, num_heads=2, num_layers=1, add_head=False, dtype=BF, device=DEV, seed=3)
  model.requires_grad_(grad)
  ids = torch.randint(1, V, (batch, length), generator=g).to(DEV)
  lens = torch.randint(0, length + 1, (batch,), generator=g)
  lens[-1] = length
  mask = (torch.arange(length)[None, :] < lens[:, None]).to(DEV)
  with torch.set_grad_enabled(grad):
    want = model(ids, seq_lens=lens.to(torch.int32).to(DEV))
    for m in (mask, mask.to(torch.uint8) * 255, mask.float()):
      assert torch.equal(model(ids.to(torch.int32), padding_mask=m), want)
    for row in range(batch) if length > 1 else ():
      bad = mask.clone()
      bad[row, 0], bad[row, length - 1] = False, True
      with pytest.raises(ValueError):
        model(ids, padding_mask=bad)
