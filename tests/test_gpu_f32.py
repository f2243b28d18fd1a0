"""The fp32-product kernels (fp32 at head dims 16, 32, 64, 128; bf16 at 16) around their tiles: 16-row blocks of a wave, 64 rows of a
workgroup, 16 or 32 streamed rows per step; every form of operand; segment and mask ranges that empty steps."""

import numpy as np
import pytest
import torch

import recml_amd
from oracle import hstu_oracle as O

pytestmark = pytest.mark.gpu


def _dev(x, dtype=None):
  t = torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")
  return t if dtype is None else t.to(dtype)


def _rel(a, b):
  return np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)


def _operands(kind, rng, B, H, L):
  """Keyword arguments for the oracle and for the package."""
  kw = dict(causal=True)
  if kind == "tables":
    kw["pos_tab"] = (rng.standard_normal((H, 2 * L - 1)) * 0.3).astype(np.float32)
    kw["ts_tab"] = (rng.standard_normal((1, 129)) * 0.3).astype(np.float32)
    kw["timestamps"] = 1_700_000_000 + np.cumsum(np.ceil(rng.exponential(3000.0, (B, L))), axis=1).astype(np.int64)
    kw["seq_lens"] = np.concatenate([[L], rng.integers(0, L + 1, B - 1)]).astype(np.int32)
  elif kind == "dense":
    i, j = np.arange(L)[None, :, None], np.arange(L)[None, None, :]
    kw["mask"] = (rng.random((B, L, L)) > 0.3) & (j <= i) & (j >= i - 40)
    kw["bias"] = (rng.standard_normal((B, L, L)) * 0.3).astype(np.float32)
    kw["causal"] = False
  elif kind == "segments":
    cuts = np.sort(rng.integers(0, L + 1, (B, 2)), axis=1)
    seg = (np.arange(L)[None] >= cuts[:, :1]).astype(np.int32) + (np.arange(L)[None] >= cuts[:, 1:])
    kw["q_segment_ids"] = kw["kv_segment_ids"] = np.where(seg == 2, 0, seg + 1).astype(np.int32)
  else:
    kw.update(causal=False, sliding_window_size=max(1, L // 3))
  gk = {dict(pos_tab="pos_bias", ts_tab="ts_bias").get(n, n): _dev(x) if isinstance(x, np.ndarray) else x for n, x in kw.items()}
  return kw, gk


@pytest.mark.parametrize("L", [1, 3, 16, 17, 63, 65, 131, 200])
@pytest.mark.parametrize("kind", ["tables", "dense", "segments", "window"])
@pytest.mark.parametrize("d,dtype", [(16, "fp32"), (32, "fp32"), (64, "fp32"), (128, "fp32"), (16, "bf16")])
def test_fp32_products(gpu, d, dtype, kind, L):
  rng = np.random.default_rng(1000 * L + d)
  B, H = 2, 3
  q, k, v, dout = (rng.standard_normal((B, L, H, d)).astype(np.float32) * 0.5 for _ in range(4))
  tol, td = 2e-5, torch.float32
  if dtype == "bf16":
    q, k, v, dout = map(O.round_bf16, (q, k, v, dout))
    tol, td = 1e-2, torch.bfloat16
  kw, gk = _operands(kind, rng, B, H, L)
  ref = O.hstu_attention_ref(q, k, v, n=9.0, alpha=0.3, **kw)
  want = O.hstu_attention_bwd_ref(q, k, v, dout, n=9.0, alpha=0.3, bias_grad=kind == "dense", **kw)
  ts = [_dev(x, td) for x in (q, k, v)]
  out = recml_amd.hstu_attention(*ts, n=9.0, alpha=0.3, **gk)
  got = recml_amd.hstu_attention_bwd(*ts, _dev(dout, td), n=9.0, alpha=0.3, bias_grad=kind == "dense", **gk)
  torch.cuda.synchronize()
  assert _rel(out.float().cpu().numpy(), ref) <= tol
  for nm, g, w in zip(("dq", "dk", "dv", "dpos", "dts", "dbias"), got, want):
    assert (g is None) == (w is None), nm
    if w is not None:
      assert _rel(g.float().cpu().numpy().reshape(w.shape), w) <= tol, nm
