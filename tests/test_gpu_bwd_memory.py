"""The scratch of a backward pass: what it asks for, and what it does where the device has not that much."""

import pytest
import torch

import recml_amd
from recml_amd import _native

pytestmark = pytest.mark.gpu
MB = 1 << 20


@pytest.fixture
def share():
  """Leaves the process so many bytes beyond those it has; the whole device again afterwards."""
  torch.cuda.synchronize()
  torch.cuda.empty_cache()                # (so that the test's tensors have pieces of their own)
  total = torch.cuda.get_device_properties(0).total_memory

  def leave(n):
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + n) / total)

  yield leave
  torch.cuda.set_per_process_memory_fraction(1.0)


def _inputs(B, L, H=8, d=128, dense=False):
  g = torch.Generator().manual_seed(L)      # (on the host, for the same reason)
  t = [torch.randn(B, L, H, d, generator=g).mul_(0.5).to(torch.bfloat16).cuda() for _ in range(4)]
  bias = (torch.randn((B, L, L) if dense else (H, 2 * L - 1), generator=g) * 0.3).cuda()
  return t, dict(bias=bias, n=float(L)) if dense else dict(pos_bias=bias)


def _gradients(t, kw, native):
  """dq, dk, dv and the bias's, by the call's autograd node or by the backward's own entry."""
  q, k, v, do = t
  if not native:
    got = recml_amd.hstu_attention_bwd(q, k, v, do, **kw, bias_grad="bias" in kw)
    return *got[:3], got[5 if "bias" in kw else 3]
  wrt = [x.detach().requires_grad_() for x in (q, k, v)]
  name = next(iter(kw))
  kw = {**kw, name: kw[name].detach().requires_grad_()}
  out = recml_amd.hstu_attention_autograd(*wrt, **kw)
  assert out.grad_fn.name() == "HstuAttentionBackward"
  return torch.autograd.grad(out, (*wrt, kw[name]), do)


def _same(a, b):
  for x, y in zip(a[:3], b[:3]):
    assert torch.equal(x, y)
  # (fp32 sums of the same terms in another order, as where the two forms of the backward are compared)
  assert float((a[3] - b[3]).abs().max()) <= 1e-4 * float(b[3].abs().max())


def _failed():
  s = torch.cuda.memory_stats()
  return s["num_alloc_retries"], s["num_ooms"]


@pytest.mark.parametrize("native,left", [(True, 232), (False, 200)])
def test_no_room_is_not_asked_for(gpu, share, native, left):
  """What the caching allocator holds is not given back for a buffer that the call can do without: 32 MB for each of dq, dk, dv (and the output),
  136 for dS."""
  t, kw = _inputs(16, 1024)
  want = _gradients(t, kw, native)
  share(left * MB)
  before = _failed()
  got = _gradients(t, kw, native)
  torch.cuda.synchronize()
  assert _failed() == before
  torch.cuda.set_per_process_memory_fraction(1.0)
  _same(got, want)


def test_room(gpu, share):
  index = torch.cuda.current_device()
  share(300 * MB)
  assert _native.has_room(index, 280 * MB) and not _native.has_room(index, 310 * MB)
  held = torch.empty(200 * MB, dtype=torch.uint8, device="cuda")
  assert not _native.has_room(index, 200 * MB) and _native.has_room(index, 96 * MB) and _native.has_room(index, 63 * MB)
  del held
  assert _native.has_room(index, 200 * MB)              # (a piece that the allocator holds)
  assert not _native.has_room(index, 203 * MB)


@pytest.mark.parametrize("native,dense,left", [(True, False, 78), (False, False, 62), (True, True, 96), (False, True, 82)])
def test_an_allocation_that_fails(gpu, share, native, dense, left):
  """Buffers below 64 MB are asked for without a look.  The call goes on without what there is no memory for, also with a dense bias's gradient (a flag of the backward's): 14 MB for each of dq, dk,
  dv (and the output), 20 for the bias's gradient, and the 38 or so of dS do not fit."""
  t, kw = _inputs(8, 768, dense=dense)
  want = _gradients(t, kw, native)
  share(left * MB)
  before = _failed()
  got = _gradients(t, kw, native)
  torch.cuda.synchronize()
  assert _failed()[1] == before[1] + 1
  torch.cuda.set_per_process_memory_fraction(1.0)
  _same(got, want)


def test_captured(gpu):
  """A backward whose scratch is large enough to be looked for, in a graph: every replay as the call itself."""
  t, kw = _inputs(16, 1024)
  want = _gradients(t, kw, False)
  side = torch.cuda.Stream()
  side.wait_stream(torch.cuda.current_stream())
  with torch.cuda.stream(side):
    _gradients(t, kw, False)
  torch.cuda.current_stream().wait_stream(side)
  torch.cuda.empty_cache()                # (no piece of that size to be found)
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    got = _gradients(t, kw, False)
  for _ in range(3):
    for x in got:
      x.fill_(7.0)
    graph.replay()
    torch.cuda.synchronize()
    _same(got, want)
    t[0].mul_(-1.0)
    want = _gradients(t, kw, False)


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
