"""Gradients of q, k and v through the projections' SiLU in the attention backward's own stores."""

import ctypes as C
from unittest import mock

import pytest
import torch

import recml_amd
from recml_amd import _lib, _lib_block

pytestmark = pytest.mark.gpu


def _case(d, lens, jagged, dtype, seed):
  """q, k, v as columns of one projection's output, as a block has them, their pre-activations and gradients laid out alike."""
  g = torch.Generator().manual_seed(seed)
  H, L = 2, max(lens)
  rows = (sum(lens),) if jagged else (len(lens), L)
  pre = (torch.randn(rows + (4, H, d), generator=g) * 1.5).to("cuda:0", dtype)
  act = torch.nn.functional.silu(pre.float()).to(dtype)
  dout = (torch.randn(rows + (H, d), generator=g) * 0.5).to("cuda:0", dtype)
  lens_t = torch.tensor(lens, dtype=torch.int32, device="cuda:0")
  kw = dict(seq_offsets=torch.cat([lens_t.new_zeros(1), lens_t.cumsum(0, dtype=torch.int32)]), max_len=L) if jagged else dict(seq_lens=lens_t)
  ts = (1_600_000_000 + torch.randint(0, 4000, rows, generator=g).cumsum(-1)).to("cuda:0")
  cols = lambda t: [t[..., i, :, :] for i in (1, 2, 3)]
  return pre, cols(act), cols(pre), dout, kw, ts, H, L


@pytest.mark.parametrize("d,lens,jagged,tables", [
    (32, [1], True, "pos"),
    (32, [33, 0, 5], False, "pos ts"),
    (64, [31, 129, 0, 256], True, "pos"),            # heads of 64 without timestamps: the kernels that take two row blocks at once
    (64, [130, 257], False, ""),
    (64, [64, 193], True, "pos ts"),
    (128, [95, 300], True, "pos ts"),
    (128, [1, 128], False, ""),
])
def test_same_as_a_pass_of_its_own(gpu, d, lens, jagged, tables):
  """The same gradients, rounded, times the same silu' : equal to a pass over the stored rows, value by value.  A pre-activation left
  out leaves that gradient as the plain backward has it."""
  pre, (q, k, v), pres, dout, kw, ts, H, L = _case(d, lens, jagged, torch.bfloat16, d)
  if "pos" in tables:
    kw["pos_bias"] = torch.randn(H, 2 * L - 1, generator=torch.Generator().manual_seed(1)).to("cuda:0") * 0.2
  if "ts" in tables:
    kw.update(timestamps=ts, ts_bias=torch.randn(H, 129, generator=torch.Generator().manual_seed(2)).to("cuda:0") * 0.2)
  lib, blk = _lib.load(), _lib_block.load()

  def run(given):
    d_uqkv = torch.full_like(pre, 7.0)
    variant = []
    call = lambda a, stream: lib.hstu_attn_bwd_silu(a, *(C.c_void_p(p.data_ptr()) if on else None for p, on in zip(pres, given)), stream)
    with mock.patch.object(lib, "hstu_attn_bwd", call):
      recml_amd.hstu_attention_bwd(q, k, v, dout, alpha=d ** -0.5, n=1024, grads_out=[d_uqkv[..., i, :, :] for i in (1, 2, 3)],
                                   _variant_out=variant, **kw)
    assert variant == ["hstu_bwd_mfma_bf16"]
    return d_uqkv

  plain = run((False, False, False))
  want = plain.clone()
  W = H * d
  rc = blk.hstu_silu_bwd(want.data_ptr() + 2 * W, 4 * W, pre.data_ptr() + 2 * W, 4 * W, pre.numel() // (4 * W), 3 * W,
                         C.c_void_p(torch.cuda.current_stream().cuda_stream))
  assert rc == 0
  assert torch.equal(run((True, True, True)), want)
  got = run((False, True, False))
  for i in range(4):
    assert torch.equal(got[..., i, :, :], (want if i == 2 else plain)[..., i, :, :])


def test_refused_without_touching_the_outputs(gpu):
  """fp32 calls, and a pre-activation off a 16-byte boundary."""
  lib = _lib.load()
  for dtype, off in ((torch.float32, 0), (torch.bfloat16, 2)):
    pre, (q, k, v), pres, dout, kw, _, _, _ = _case(32, [40], True, dtype, 3)
    d_uqkv = torch.full_like(pre, 7.0)
    call = lambda a, stream: lib.hstu_attn_bwd_silu(a, *(C.c_void_p(p.data_ptr() + off) for p in pres), stream)
    with mock.patch.object(lib, "hstu_attn_bwd", call), pytest.raises(ValueError, match="activation|aligned"):
      recml_amd.hstu_attention_bwd(q, k, v, dout, grads_out=[d_uqkv[..., i, :, :] for i in (1, 2, 3)], **kw)
    torch.cuda.synchronize()
    assert bool((d_uqkv == 7.0).all())
