"""The timestamp table's gradient where a tile's keys lie in two neighbouring buckets: each bucket's sum is made of its own pairs'
terms alone, whatever the other bucket's are."""

import numpy as np
import pytest
import torch

import recml_amd
from oracle import hstu_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("far", [2.0 ** 20, float("inf")])
def test_near_bucket_keeps_its_own_sum(gpu, d, far):
  """Keys 0..15 and 16..31 share a tile and lie 13000 and 10000 seconds before the rows that follow: buckets 31 and 30.  The far
  keys' values, and with them their pairs' dS, are larger by 2^20, or infinite.  Bound: the near sum's own terms carry errors of a
  few 2^-22 of their magnitudes (fp32 products and sums, the hardware's exponential), which cancel to a tenth at most; one as what is
  left of both buckets' total is off by several percent."""
  rng = np.random.default_rng(5)
  B, L, H = 1, 64, 1
  q, k, v, dout = (O.round_bf16(rng.standard_normal((B, L, H, d)).astype(np.float32) * 0.5) for _ in range(4))
  ts = np.concatenate([np.zeros(16), np.full(16, 3000), np.full(32, 13000)]).astype(np.int64)[None] + 1_600_000_000
  tab = (rng.standard_normal((H, 129)) * 0.3).astype(np.float32)
  want = O.hstu_attention_bwd_ref(q, k, v, dout, timestamps=ts, ts_tab=tab)[4]      # (a bucket's sum does not depend on another's values)
  assert want[0, 30] != 0 and want[0, 31] != 0
  v = v.copy()
  v[:, :16] = v[:, :16] * 2.0 ** 20 if np.isfinite(far) else far
  dev = lambda x, dt=None: torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0").to(dt or torch.from_numpy(np.ascontiguousarray(x)).dtype)
  bf = torch.bfloat16
  variant = []
  got = recml_amd.hstu_attention_bwd(dev(q, bf), dev(k, bf), dev(v, bf), dev(dout, bf), timestamps=dev(ts), ts_bias=dev(tab),
                                     _variant_out=variant)[4].cpu().numpy()
  assert variant == ["hstu_bwd_mfma_bf16"]
  assert abs(got[0, 30] - want[0, 30]) <= 1e-3 * abs(want[0, 30])
  if np.isfinite(far):
    assert abs(got[0, 31] - 2.0 ** 20 * want[0, 31]) <= 1e-3 * abs(2.0 ** 20 * want[0, 31])
  else:
    assert not np.isfinite(got[0, 31])
