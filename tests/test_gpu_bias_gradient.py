"""The dense bias's gradient, which has a kernel of its own where there are tiles enough, against the fp32 kernels on the same values."""

import pytest
import torch

import recml_amd
from recml_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _call(B, L, H, d, kind, seed=0):
  g = torch.Generator().manual_seed(B * L + H + seed)
  q, k, v, dout = ((torch.randn(B, L, H, d, generator=g) * 0.5).to(DEV, torch.bfloat16) for _ in range(4))
  lens = torch.randint(1, L + 1, (B,), generator=g)
  lens[0] = L
  i = torch.arange(L)
  kw = dict(alpha=d**-0.5, n=64.0, bias=(torch.randn((L, L) if kind == "shared" else (B, L, L), generator=g) * 0.3).to(DEV))
  if kind in ("mask", "shared"):
    keep = (i[None, :, None] >= i[None, None, :]) & (i[None, None, :] < lens[:, None, None]) & (torch.rand(B, L, L, generator=g) < 0.9)
    keep[-1, 100:400] = False            # rows and whole tiles without a key
    kw.update(mask=keep.to(DEV), causal=False)
  elif kind == "lengths":
    kw.update(seq_lens=lens.int().to(DEV))
  elif kind == "full":
    kw.update(causal=False)
  else:
    kw.update(seq_lens=lens.int().to(DEV), sliding_window_size=L // 5, dropout_p=0.2, dropout_seed=11)
  return q, k, v, dout, kw


@pytest.mark.parametrize("B,L,H,d,kind", [
    (12, 513, 3, 64, "mask"),            # rows of no whole 16 bytes, one row and one key past the tiles
    (3, 1024, 2, 128, "mask"),           # two stages a head
    (12, 520, 2, 32, "lengths"),
    (5, 900, 3, 64, "window"),           # with dropout
    (12, 512, 1, 64, "full"),
    (1, 1800, 2, 128, "shared"),
    # short rows of many sequences: one step, less than a tile, odd lengths
    (64, 30, 2, 64, "mask"), (64, 31, 2, 128, "lengths"), (100, 17, 1, 32, "window"),
    (64, 100, 2, 32, "lengths"), (40, 97, 2, 128, "mask"), (33, 127, 2, 64, "window"),
    (16, 201, 3, 64, "window"), (12, 267, 2, 128, "mask"), (16, 155, 4, 32, "full"),
    (14, 150, 3, 64, "lengths"), (13, 150, 3, 64, "lengths"),              # 28 tiles of 128 x 64 a head, and less: added by the dQ kernel
    (64, 60, 1, 128, "mask"), (63, 60, 1, 128, "mask"),                  # 64 tiles, and less
])
def test_against_fp32(gpu, B, L, H, d, kind):
  """Both form S and dP from the same values in fp32 sums of d terms and add H of their products in fp32: relative differences of some
  2^-24 sqrt(d H), 2e-6, and of single values up to 2^-24 d of the largest."""
  q, k, v, dout, kw = _call(B, L, H, d, kind)
  variant = []
  got = recml_amd.hstu_attention_bwd(q, k, v, dout, bias_grad=True, _variant_out=variant, **kw)[5]
  assert variant == ["hstu_bwd_mfma_bf16"]
  want = recml_amd.hstu_attention_bwd(q.float(), k.float(), v.float(), dout.float(), bias_grad=True, **kw)[5]
  assert bool(torch.isfinite(got).all())
  assert bool(((got == 0) >= (want == 0)).all())       # nothing where no pair is kept
  diff = (got - want).double()
  assert float(diff.norm()) <= 1e-5 * float(want.double().norm())
  assert float(diff.abs().max()) <= 2.0**-15 * float(want.abs().max())
  again = recml_amd.hstu_attention_bwd(q, k, v, dout, bias_grad=True, **kw)[5]
  tiles = B * ((L + 127) // 128) * ((L + 63) // 64)
  if tiles >= max(64, 28 * H):
    assert torch.equal(got, again)
  else:      # (the dQ kernel's additions come in any order: H - 1 roundings of at most the terms' magnitudes' sum on either side)
    assert float((got - again).abs().max()) <= 2 * H * 2.0**-24 * H * float(got.abs().max())


@pytest.mark.parametrize("B,L", [(12, 520), (2, 200)])
def test_added_to_what_is_there(gpu, monkeypatch, B, L):
  """A caller that does not ask for it to be written: it is added to, with the kernel and without."""
  q, k, v, dout, kw = _call(B, L, 2, 64, "mask" if L == 520 else "lengths")
  want = recml_amd.hstu_attention_bwd(q, k, v, dout, bias_grad=True, **kw)[5]
  monkeypatch.setattr(_lib, "BWD_WRITE_BIAS_GRADIENT", 0)
  monkeypatch.setattr(torch, "empty", torch.ones)
  got = recml_amd.hstu_attention_bwd(q, k, v, dout, bias_grad=True, **kw)[5]
  assert float((got - want - 1.0).abs().max()) <= 2.0**-22 * float(1 + want.abs().max()) * 2
