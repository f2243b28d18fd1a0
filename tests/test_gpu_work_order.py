"""The work list's order: every tile of every sequence is done once, whatever the lengths and wherever the part of the list that goes by
tile index begins."""

import ctypes

import pytest
import torch

import recml_amd
from recml_amd import _lib, hstu_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,H,d,kind,jagged", [
    (1, 513, 8, 64, "full", True),               # one sequence, the shortest that has a list
    (40, 1100, 16, 32, "full", True),            # 360 tiles, 128 (forward) and 256 (backward) of them at the list's end by tile index
    (40, 1100, 16, 32, "mixed", True),
    (40, 1100, 16, 32, "mixed", False),          # (padded: the rows past a length are tiles of their own, stored as zeros)
    (6, 2300, 8, 128, "mixed", True),            # all by tile index
    (24, 640, 2, 64, "mixed", True),             # fewer heads than XCDs
    (40, 1100, 12, 32, "mixed", True),           # head counts dealt to the XCDs in groups of items
    (90, 900, 3, 64, "mixed", False),
    (31, 1000, 6, 128, "full", True),
    (9, 700, 12, 32, "none", True),              # no tokens but those of the last sequence
    (16, 500, 4, 64, "mixed", True),             # no list: the backward takes all sequences' last tiles first
    (15, 500, 3, 128, "mixed", False),           # the same with XCDs that have one sequence less than others
    (1030, 530, 1, 32, "mixed", True),           # more sequences than are ordered at a time
])
@pytest.mark.parametrize("causal", [True, False])
def test_every_tile_once(gpu, B, L, H, d, kind, jagged, causal):
  """The backward of the batch equals, bit by bit, that of each sequence alone: its row gradients do not depend on the list.  The
  forward's do where a tile's keys are split: sums of fp32 terms in another order, rounded to bf16: a last place of the row's largest
  values, 2^-7 of them.  Outputs start as NaN, so that a tile left out shows."""
  g = torch.Generator().manual_seed(B + L)
  if kind == "full":
    lens = torch.full((B,), L)
  elif kind == "none":
    lens = torch.zeros(B, dtype=torch.long)
    lens[-1] = L
  else:
    lens = torch.randint(0, L + 1, (B,), generator=g)
    for i, n in enumerate((0, 1, 127, 128, 129, L)):
      lens[(7 * i) % B] = n
  off = torch.cat([torch.zeros(1, dtype=torch.long), lens.cumsum(0)])
  rows = (int(off[-1]),) if jagged else (B, L)
  q, k, v, dout = ((torch.randn(rows + (H, d), generator=g) * 0.5).to("cuda:0", torch.bfloat16) for _ in range(4))
  pos = (torch.randn(H, 2 * L - 1, generator=g) * 0.2).to("cuda:0")
  kw = dict(causal=causal, alpha=d ** -0.5, n=1024, pos_bias=pos)
  batch = dict(seq_offsets=off.int().to("cuda:0"), max_len=L) if jagged else dict(seq_lens=lens.int().to("cuda:0"))
  nan = lambda t: torch.full_like(t, float("nan"))
  out = recml_amd.hstu_attention(q, k, v, out=nan(q), **batch, **kw)
  grads = [nan(q) for _ in range(3)]
  variant = []
  recml_amd.hstu_attention_bwd(q, k, v, dout, grads_out=grads, _variant_out=variant, **batch, **kw)
  assert variant == ["hstu_bwd_mfma_bf16"]
  for b in range(B) if B <= 40 else range(0, B, 41):
    n = int(lens[b])
    at = slice(int(off[b]), int(off[b]) + n) if jagged else (b, slice(0, n))
    if not jagged:
      for t in (out, *grads):
        assert bool((t[b, n:] == 0).all())
    if n == 0:
      continue
    one = dict(seq_offsets=torch.tensor([0, n], dtype=torch.int32, device="cuda:0"), max_len=L)
    want = recml_amd.hstu_attention(q[at], k[at], v[at], **one, **kw).float()
    scale = want.abs().amax((-1, -2), keepdim=True)
    assert bool(((out[at].float() - want).abs() <= 2.0 ** -7 * scale).all())
    for got, ref in zip(grads, recml_amd.hstu_attention_bwd(q[at], k[at], v[at], dout[at], table_grads=False, **one, **kw)):
      assert torch.equal(got[at], ref)
  if B > 40:
    for t in (out, *grads):
      assert bool(torch.isfinite(t).all())


def test_without_room_for_a_list(gpu):
  """Head counts that neither divide 8 nor are divided by it: a call without a workspace, or with too little for the list, is taken."""
  g = torch.Generator().manual_seed(3)
  lens, L, H, d = [900, 0, 300, 1024] + 18 * [40], 1024, 12, 64
  q, k, v = ((torch.randn(sum(lens), H, d, generator=g) * 0.5).to("cuda:0", torch.bfloat16) for _ in range(3))
  off = torch.tensor([0] + lens, device="cuda:0").cumsum(0).int()
  want = recml_amd.hstu_attention(q, k, v, seq_offsets=off, max_len=L).float()
  lib = _lib.load()
  stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
  for room in (0, 256):
    out = torch.full_like(q, float("nan"))
    args, keep = hstu_ops.build_args(q, k, v, out, seq_offsets=off, max_len=L)
    assert args.workspace_bytes > 256
    args.workspace_bytes = room
    args.workspace = args.workspace if room else None
    assert lib.hstu_attn_fwd(ctypes.byref(args), stream) == 0
    assert bool(((out.float() - want).abs() <= 2.0 ** -7 * want.abs().amax((-1, -2), keepdim=True)).all())
    bwd = _lib.HstuAttnBwdArgs(struct_size=ctypes.sizeof(_lib.HstuAttnBwdArgs), version=_lib.ABI_VERSION, fwd=args)
    grads = [torch.full_like(q, float("nan")) for _ in range(3)]
    bwd.dout, bwd.dq, bwd.dk, bwd.dv = v.data_ptr(), *(t.data_ptr() for t in grads)
    assert lib.hstu_attn_bwd_variant(ctypes.byref(bwd)) == b"hstu_bwd_mfma_bf16"
    assert lib.hstu_attn_bwd(ctypes.byref(bwd), stream) == 0
    for got, ref in zip(grads, recml_amd.hstu_attention_bwd(q, k, v, v, seq_offsets=off, max_len=L)):
      assert torch.equal(got, ref)
    torch.cuda.synchronize()
    del keep


def _rows_alone(kind, B, L, H, d, g, dev="cuda:0"):
  """A batch with one kind of operand beside q, k and v, and a function that gives the operand's part for one sequence."""
  q, k, v, dout = ((torch.randn(B, L, H, d, generator=g) * 0.5).to(dev, torch.bfloat16) for _ in range(4))
  lens = torch.randint(1, L + 1, (B,), generator=g)
  lens[0] = L
  i = torch.arange(L)
  if kind == "dense":
    mask = ((i[None, :, None] >= i[None, None, :]) & (i[None, None, :] < lens[:, None, None])).to(dev)
    bias = (torch.randn(B, L, L, generator=g) * 0.2).to(dev)
    return q, k, v, dout, lambda at: dict(mask=mask[at], bias=bias[at], causal=False)
  ids = torch.where(i[None] < (lens // 2)[:, None], 1, torch.where(i[None] < lens[:, None], 2, 0)).int().to(dev)
  return q, k, v, dout, lambda at: dict(q_segment_ids=ids[at], kv_segment_ids=ids[at])


@pytest.mark.parametrize("kind", ["dense", "segments"])
@pytest.mark.parametrize("B,L,H,d", [(30, 1000, 3, 64), (12, 1024, 6, 128), (24, 640, 12, 32), (24, 640, 2, 64)])
def test_every_tile_once_with_other_operands(gpu, kind, B, L, H, d):
  """As above where the batch brings a dense mask and bias, or segment ids, at head counts on either side of the XCDs' eight."""
  g = torch.Generator().manual_seed(B * L + H)
  q, k, v, dout, part = _rows_alone(kind, B, L, H, d, g)
  kw = dict(alpha=d ** -0.5, n=1024)
  nan = lambda t: torch.full_like(t, float("nan"))
  whole = slice(None)
  out = recml_amd.hstu_attention(q, k, v, out=nan(q), **part(whole), **kw)
  grads, variant = [nan(q) for _ in range(3)], []
  recml_amd.hstu_attention_bwd(q, k, v, dout, grads_out=grads, _variant_out=variant, **part(whole), **kw)
  assert variant == ["hstu_bwd_mfma_bf16"]
  for b in range(0, B, 3):
    at = slice(b, b + 1)
    want = recml_amd.hstu_attention(q[at], k[at], v[at], **part(at), **kw).float()
    assert bool(((out[at].float() - want).abs() <= 2.0 ** -7 * want.abs().amax((-1, -2), keepdim=True)).all())
    for got, ref in zip(grads, recml_amd.hstu_attention_bwd(q[at], k[at], v[at], dout[at], **part(at), **kw)):
      assert torch.equal(got[at], ref)
  for t in (out, *grads):
    assert bool(torch.isfinite(t).all())


@pytest.mark.parametrize("H", [2, 3, 6, 12])
def test_every_tile_once_in_fp8(gpu, H):
  """The forward's list with 8-bit queries and keys, against each sequence alone."""
  B, L, d = 20, 1200, 128
  g = torch.Generator().manual_seed(H)
  lens = torch.randint(1, L + 1, (B,), generator=g)
  off = torch.cat([torch.zeros(1, dtype=torch.long), lens.cumsum(0)])
  q, k = ((torch.randn(int(off[-1]), H, d, generator=g) * 0.5).to("cuda:0").to(torch.float8_e4m3fn) for _ in range(2))
  v = torch.randn(int(off[-1]), H, d, generator=g).to("cuda:0", torch.bfloat16)
  pos = (torch.randn(H, 2 * L - 1, generator=g) * 0.2).to("cuda:0")
  kw = dict(alpha=d ** -0.5, n=1024, pos_bias=pos)
  out = torch.full_like(v, float("nan"))
  recml_amd.hstu_attention(q, k, v, out=out, seq_offsets=off.int().to("cuda:0"), max_len=L, **kw)
  for b in range(B):
    at = slice(int(off[b]), int(off[b + 1]))
    one = dict(seq_offsets=torch.tensor([0, int(lens[b])], dtype=torch.int32, device="cuda:0"), max_len=L)
    want = recml_amd.hstu_attention(q[at], k[at], v[at], **one, **kw).float()
    assert bool(((out[at].float() - want).abs() <= 2.0 ** -7 * want.abs().amax((-1, -2), keepdim=True)).all())
