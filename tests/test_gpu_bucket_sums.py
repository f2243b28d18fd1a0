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


@pytest.mark.parametrize("d,L,causal,window,lens", [
    (32, 1, True, None, [1]),
    (64, 33, True, None, [33, 32]),                  # the second wave's one row; a wave's last block is its first
    (128, 300, True, None, [300, 129, 97, 5]),       # the rings of diagonal sums begin again at 256
    (64, 700, False, None, [700, 257]),              # every wave ends at the same step: what waits is handed on after the loop
    (128, 520, True, 40, [520, 383]),                # a band narrower than a tile, starting and ending at another step in each wave
    (32, 420, False, 130, [420, 31]),
])
def test_table_sums_are_complete(gpu, d, L, causal, window, lens):
  """q = k = 0 and both tables 0: every logit is 0 and f' a half, dS half of a small whole number, and every sum of them exact in
  fp32, in whatever order it is made.  So both tables' gradients are equal to the reference's, bit by bit.  An item about every hour:
  one bucket, two and more than two to a block, and a bucket's run that goes on from one block to the next."""
  rng = np.random.default_rng(L)
  B, H = len(lens), 2
  zero = np.zeros((B, L, H, d), np.float32)
  v, dout = (rng.integers(-1, 2, (B, L, H, d)).astype(np.float32) for _ in range(2))
  ts = 1_600_000_000 + np.cumsum(np.ceil(rng.exponential(3600.0, (B, L))).astype(np.int64), 1)
  pos, tab = np.zeros((H, 2 * L - 1), np.float32), np.zeros((H, 129), np.float32)
  lens = np.array(lens, np.int32)
  want = O.hstu_attention_bwd_ref(zero, zero, v, dout, causal=causal, sliding_window_size=window, seq_lens=lens, n=1024, pos_tab=pos,
                                  timestamps=ts, ts_tab=tab)
  dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")
  for dtype, pos_, ts_ in ((torch.bfloat16, True, True), (torch.bfloat16, True, False), (torch.bfloat16, False, True), (torch.float32, True, True)):
    kw = dict(pos_bias=dev(pos)) if pos_ else {}
    kw.update(dict(timestamps=dev(ts), ts_bias=dev(tab)) if ts_ else {})
    variant = []
    got = recml_amd.hstu_attention_bwd(dev(zero).to(dtype), dev(zero).to(dtype), dev(v).to(dtype), dev(dout).to(dtype), causal=causal,
                                       sliding_window_size=window, seq_lens=dev(lens), n=1024, _variant_out=variant, **kw)
    assert dtype == torch.float32 or variant == ["hstu_bwd_mfma_bf16"]
    for g, w, given in ((got[3], want[3], pos_), (got[4], want[4], ts_)):
      assert (g is not None) == given
      if given:
        np.testing.assert_array_equal(g.cpu().numpy(), np.asarray(w, np.float32))
