"""The backward with the logits' gradients kept between its two kernels against the one that forms them twice, in bf16 and fp32: what decides is
the workspace that the caller brings, and both give the same bits (but for dQ where a timestamp table stands alone, dK and dV of d = 128 without tables
and segment ids, and the tables' gradients: fp32 operations in another order)."""

import ctypes as C

import numpy as np
import pytest
import torch

import recml_amd
from recml_amd import _lib

pytestmark = pytest.mark.gpu


def _least(args):
  """Bytes that the kernels need that each form dS for themselves.  (The forward's question knows no flag of the backward's.)"""
  f = args._obj.fwd
  flags, f.flags = f.flags, f.flags & ~_lib.BWD_WRITE_BIAS_GRADIENT
  n = _lib.load().hstu_attn_fwd_workspace_bytes(C.byref(f))
  f.flags = flags
  return n


@pytest.fixture
def handed_on(monkeypatch):
  """For each backward call whether something was written behind what `_least` says: only blocks of dS are."""
  lib, seen = _lib.load(), []
  call = lib.hstu_attn_bwd

  def watched(args, stream):
    f, least = args._obj.fwd, _least(args)
    scratch = torch.full((max(f.workspace_bytes, 1),), 0xA5, dtype=torch.uint8, device="cuda")
    if f.workspace_bytes:
      f.workspace = scratch.data_ptr()
    rc = call(args, stream)
    seen.append(bool((scratch[least:f.workspace_bytes] != 0xA5).any()))
    return rc

  monkeypatch.setattr(lib, "hstu_attn_bwd", watched)
  return seen


def _case(dtype, d, L, H, lens, *, jagged, pos, ts, seg, B):
  g = torch.Generator(device="cuda").manual_seed(d + L)
  n = np.array(lens if lens is not None else [L] * B, np.int32)
  shape = (int(n.sum()), H, d) if jagged else (B, L, H, d)
  q, k, v, do = (torch.randn(shape, device="cuda", generator=g).mul_(0.5).to(dtype) for _ in range(4))
  kw = {}
  if jagged:
    kw.update(seq_offsets=torch.from_numpy(np.concatenate([[0], np.cumsum(n)]).astype(np.int32)).cuda(), max_len=L)
  elif lens is not None:
    kw["seq_lens"] = torch.from_numpy(n).cuda()
  if pos:
    kw["pos_bias"] = torch.randn(H, 2 * L - 1, device="cuda", generator=g) * 0.3
  if ts:
    gaps = torch.randint(1, 7200, (shape[0],) if jagged else (B, L), device="cuda", generator=g)
    kw.update(timestamps=1_600_000_000 + torch.cumsum(gaps, -1), ts_bias=torch.randn(129, device="cuda", generator=g) * 0.3)
  if seg:
    ids = torch.randint(0, 3, (B, L), device="cuda", generator=g).sort(-1).values.to(torch.int32)
    kw.update(q_segment_ids=ids, kv_segment_ids=ids)
  return q, k, v, do, kw


_FORMS = [
    (128, 2, 256, 8, None, {}),                                                             # whole tiles; the other side: the stream
    (128, 5, 420, 2, [420, 129, 33, 1, 256], dict(jagged=1, pos=1, ts=1)),
    (128, 5, 420, 4, [0, 420, 31, 32, 97], dict(pos=1)),                                    # a sequence without a token, block edges
    (128, 3, 300, 3, [300, 128, 5], dict(ts=1, causal=False)),                              # rectangular blocks, no list
    (128, 2, 400, 2, [400, 333], dict(pos=1, sliding_window_size=37)),
    (128, 2, 400, 2, None, dict(causal=False, sliding_window_size=150)),
    (128, 2, 333, 2, [333, 290], dict(sliding_window_size=0)),                               # bands of one block a row and of two, a row more than the last
    (128, 3, 333, 2, [333, 64, 33], dict(jagged=1, pos=1, ts=1, sliding_window_size=31)),
    (64, 3, 420, 2, [420, 97, 300], dict(jagged=1, pos=1, sliding_window_size=32, causal=False)),
    (64, 2, 420, 2, [420, 333], dict(pos=1, ts=1, sliding_window_size=33)),
    (128, 3, 260, 2, None, dict(seg=1)),
    (128, 3, 300, 2, [300, 200, 64], dict(jagged=1, pos=1, ts=1, dropout_p=0.3, dropout_seed=7)),
    (64, 5, 420, 8, [420, 129, 33, 1, 256], dict(jagged=1, pos=1, ts=1)),
    (64, 2, 200, 4, [200, 100], dict(pos=1, causal=False)),
    (64, 3, 260, 2, None, dict(seg=1)),
    (32, 5, 420, 2, [420, 129, 33, 1, 256], dict(jagged=1, ts=1)),
    (32, 2, 333, 1, None, dict(pos=1, ts=1, sliding_window_size=50)),
    (64, 4, 300, 4, [300, 129, 33, 1], dict(jagged=1)),                                     # the order of the kept form on both sides
    (32, 4, 300, 4, [300, 129, 33, 1], dict(jagged=1, pos=1, ts=1)),
]


@pytest.mark.parametrize("d,form", [(64, {}), (64, dict(seg=1)), (64, dict(causal=False)), (64, dict(dropout_p=0.2, dropout_seed=3)), (32, dict(pos=1, ts=1)),
                                    (32, dict(pos=1, ts=1, causal=False)), (32, dict(jagged=1, pos=1, ts=1, sliding_window_size=40))])
@pytest.mark.parametrize("B,L,H", [(3, 420, 2), (100, 60, 24), (33, 100, 32)])
def test_both_orders_of_products(gpu, monkeypatch, d, form, B, L, H):
  """With dS formed twice the order of dK/dV's products and vector part goes by whether the longest tile or the work lasts longer (the first batch;
  the other two): the same bits of all gradients as with the order of the kept form."""
  opt = dict(form)
  form = {x: opt.pop(x, 0) for x in ("jagged", "pos", "ts", "seg")}
  rng = np.random.default_rng(B)
  q, k, v, do, kw = _case(torch.bfloat16, d, L, H, None if form["seg"] else [L] + [int(x) for x in rng.integers(0, L + 1, B - 1)], B=B, **form)
  kw.update(opt)
  lib = _lib.load()
  a = recml_amd.hstu_attention_bwd(q, k, v, do, **kw)
  monkeypatch.setattr(lib, "hstu_attn_bwd_workspace_bytes", lambda args: lib.hstu_attn_fwd_workspace_bytes(C.byref(args._obj.fwd)))
  b = recml_amd.hstu_attention_bwd(q, k, v, do, **kw)
  for name, x, y in zip(("dq", "dk", "dv"), a, b):
    assert torch.equal(x, y), name


@pytest.mark.parametrize("d", [128, 64, 32])
@pytest.mark.parametrize("form", [dict(jagged=1, pos=1, ts=1), dict(jagged=1, ts=1), dict(pos=1), dict(jagged=1, pos=1, ts=1, dropout_p=0.3, dropout_seed=5),
                                  dict(pos=1, ts=1, sliding_window_size=70), dict(pos=1, causal=False)])
def test_frozen_tables(gpu, monkeypatch, d, form):
  """No table's gradient wanted: an instance without the sums for them, and the same bits of dq, dk and dv."""
  opt = dict(form)
  form = {x: opt.pop(x, 0) for x in ("jagged", "pos", "ts", "seg")}
  q, k, v, do, kw = _case(torch.bfloat16, d, 420, 4, [420, 129, 33, 1, 0, 256], B=6, **form)
  kw.update(opt)
  want = recml_amd.hstu_attention_bwd(q, k, v, do, **kw)
  got = recml_amd.hstu_attention_bwd(q, k, v, do, table_grads=False, **kw)
  assert got[3] is None and got[4] is None
  for name, x, y in zip(("dq", "dk", "dv"), got, want):
    assert torch.equal(x, y), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,B,L,H,lens,opt", _FORMS)
def test_kept_and_formed_twice_agree(gpu, monkeypatch, handed_on, dtype, d, B, L, H, lens, opt):
  if dtype == torch.float32:
    H *= 64 if "sliding_window_size" in opt else 16          # (small fp32 calls keep nothing: below 2e8 bytes of blocks times the head dim)
  opt = dict(opt)
  form = {x: opt.pop(x, 0) for x in ("jagged", "pos", "ts", "seg")}
  q, k, v, do, kw = _case(dtype, d, L, H, lens, B=B, **form)
  kw.update(opt)
  lib = _lib.load()
  best, least = [], []
  whole = lib.hstu_attn_bwd_workspace_bytes

  def kept(args):
    best.append(whole(args))
    return best[-1]

  def formed_twice(args):          # (a little more than the least, too: the room is not enough, and nothing is kept)
    least.append(_least(args))
    return least[-1] + 4096

  monkeypatch.setattr(lib, "hstu_attn_bwd_workspace_bytes", kept)
  a = recml_amd.hstu_attention_bwd(q, k, v, do, **kw)
  again = recml_amd.hstu_attention_bwd(q, k, v, do, **kw)
  monkeypatch.setattr(lib, "hstu_attn_bwd_workspace_bytes", formed_twice)
  b = recml_amd.hstu_attention_bwd(q, k, v, do, **kw)
  assert best[0] > least[0] + 4096
  assert handed_on == [True, True, False]
  for name, x, y, z in zip(("dq", "dk", "dv"), a, b, again):
    assert torch.equal(x, z), name
    if dtype == torch.bfloat16 and ((name == "dq" and form["ts"] and not form["pos"]) or (name != "dq" and d == 128 and not (form["pos"] or form["ts"] or form["seg"]))):
      # dq: a logit and its timestamp bias added with one rounding or two, which turns a bf16 rounding of dS now and then; dk, dv: fp32 sums in
      # two halves or in one.  Either shows as a last bit of single elements: far below the rounding of all of them, 2^-9 of the norm.
      assert float((x.float() - y.float()).norm()) <= 2.0 ** -9 * float(y.float().norm()), name
    else:
      assert torch.equal(x, y), name
  # the tables' gradients are fp32 sums of the same terms in another order: an entry's error is below (its terms) x 2^-24 x the sum of
  # their magnitudes, at most B L H terms, whose sum stays within a few times the largest entry here; 1e-4 of it covers both sides' orders
  for name, x, y in zip(("dpos", "dts"), a[3:], b[3:]):
    assert (x is None) == (y is None), name
    if x is not None:
      assert float((x - y).abs().max()) <= 1e-4 * float(y.abs().max()), name


@pytest.mark.parametrize("d", [128, 64, 32])
@pytest.mark.parametrize("B,L,Lkv,bias", [(2, 200, 200, True), (2, 77, 77, False), (3, 50, 130, True), (2, 130, 50, False)])
def test_fp32_with_dense_operands(gpu, monkeypatch, handed_on, d, B, L, Lkv, bias):
  """A mask and a dense bias, keys and queries of different lengths: blocks without a kept pair are neither written nor read."""
  g = torch.Generator(device="cuda").manual_seed(d + L)
  H = 160
  q, do = (torch.randn(B, L, H, d, device="cuda", generator=g) * 0.5 for _ in range(2))
  k, v = (torch.randn(B, Lkv, H, d, device="cuda", generator=g) * 0.5 for _ in range(2))
  mask = torch.rand(B, L, Lkv, device="cuda", generator=g) < 0.3
  mask[:, 16:48] = False
  mask[:, :, 16:32] = False
  kw = dict(mask=mask, causal=False, n=float(L))
  if bias:
    kw.update(bias=torch.randn(B, L, Lkv, device="cuda", generator=g) * 0.3, bias_grad=True)
  lib = _lib.load()
  whole, best = lib.hstu_attn_bwd_workspace_bytes, []
  monkeypatch.setattr(lib, "hstu_attn_bwd_workspace_bytes", lambda args: best.append(whole(args)) or best[-1])
  a = recml_amd.hstu_attention_bwd(q, k, v, do, **kw)
  assert best[0] > 0
  monkeypatch.setattr(lib, "hstu_attn_bwd_workspace_bytes", lambda args: 0)
  b = recml_amd.hstu_attention_bwd(q, k, v, do, **kw)
  assert handed_on == [True, False]
  for x, y in zip(a[:3], b[:3]):
    assert torch.equal(x, y)
  if bias:      # (the heads' terms added by atomics in any order: H - 1 roundings of at most the terms' magnitudes' sum on either side)
    assert float((a[5] - b[5]).abs().max()) <= 2 * H * 2.0 ** -24 * H * float(a[5].abs().max())


@pytest.mark.parametrize("d", [128, 64, 32])
@pytest.mark.parametrize("B,L,lens,bias,how", [
    (3, 420, [420, 129, 33], True, "causal"), (40, 60, None, True, "random"), (40, 70, [70] * 20 + [33] * 20, True, "causal"), (2, 300, None, True, "random"), (2, 300, [300, 128], False, "random"), (9, 513, None, True, "none"),
    (1, 1100, None, False, "band"),
])
def test_bf16_with_dense_operands(gpu, monkeypatch, handed_on, d, B, L, lens, bias, how):
  """Blocks of the mask's tiles without a kept pair are neither written nor read."""
  g = torch.Generator(device="cuda").manual_seed(d + L)
  H = 2
  q, k, v, do = (torch.randn(B, L, H, d, device="cuda", generator=g).mul_(0.5).to(torch.bfloat16) for _ in range(4))
  i, j = torch.arange(L, device="cuda")[:, None], torch.arange(L, device="cuda")[None, :]
  mask = {"causal": (i >= j).expand(B, L, L), "band": (i - j).abs() < 40, "none": None,
          "random": torch.rand(B, L, L, device="cuda", generator=g) < 0.3}[how]
  if how == "random":
    mask[:, 32:64] = False
    mask[:, 128:256, :128] = False
    mask[:, :, 64:96] = False
  kw = dict(causal=how == "none", n=float(L))
  if mask is not None:
    kw["mask"] = mask.contiguous()
  if lens is not None:
    kw["seq_lens"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
  if bias:
    kw.update(bias=torch.randn(B, L, L, device="cuda", generator=g) * 0.3)
  lib = _lib.load()
  whole, best = lib.hstu_attn_bwd_workspace_bytes, []
  monkeypatch.setattr(lib, "hstu_attn_bwd_workspace_bytes", lambda args: best.append(whole(args)) or best[-1])
  a = recml_amd.hstu_attention_bwd(q, k, v, do, **kw)
  monkeypatch.setattr(lib, "hstu_attn_bwd_workspace_bytes", _least)
  b = recml_amd.hstu_attention_bwd(q, k, v, do, **kw)
  assert handed_on == [True, False]
  assert best[0] > B * H * L * L       # (two bytes for each of half the pairs at least)
  for name, x, y in zip(("dq", "dk", "dv"), a, b):
    assert torch.equal(x, y), name
  if not bias:
    return
  # with the bias's gradient: apart where there are tiles enough, else added by the kernel that forms dS for itself
  apart = B * ((L + 127) // 128) * ((L + 63) // 64) >= 64
  twice = recml_amd.hstu_attention_bwd(q, k, v, do, bias_grad=True, **kw)
  monkeypatch.setattr(lib, "hstu_attn_bwd_workspace_bytes", whole)
  once = recml_amd.hstu_attention_bwd(q, k, v, do, bias_grad=True, **kw)
  assert handed_on[2:] == [False, apart]
  for name, x, y, z in zip(("dq", "dk", "dv"), a, once, twice):
    assert torch.equal(x, y) and torch.equal(x, z), name
  # (two heads' terms of a pair added in fp32 in either order: one rounding)
  assert bool(torch.isfinite(once[5]).all()) and float((once[5] - twice[5]).abs().max()) <= 2.0 ** -23 * float(twice[5].abs().max())
