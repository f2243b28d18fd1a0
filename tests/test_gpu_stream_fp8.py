"""The hand-scheduled stream with 8-bit queries and keys (d = 128): the bits of the compiler-scheduled block code, on sequences
around the stream's four-step rounds, with and without the position table, and the oracle's values."""

import numpy as np
import pytest
import torch

from recml_amd import _lib, hstu_ops
from oracle import hstu_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pos", [False, True])
@pytest.mark.parametrize("causal,jagged", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("lens,H", [([2048, 1655, 1000, 641, 640, 513, 385, 384, 383, 129, 16, 1], 8), ([900, 512], 2)])
def test_stream_of_8_bit_operands(gpu, lens, H, causal, jagged, pos):
  g = torch.Generator(device="cuda:0").manual_seed(7)
  lens = np.asarray(lens, np.int32)
  L, d = int(lens.max()), 128
  kw = dict(max_len=L, n=L, causal=causal)
  if jagged:
    kw["seq_offsets"] = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).to("cuda:0")
    shape = (int(lens.sum()), H, d)
  else:
    kw["seq_lens"] = torch.from_numpy(lens).to("cuda:0")
    shape = (len(lens), L, H, d)
  q, k = (torch.randn(shape, device="cuda:0", generator=g).to(torch.float8_e4m3fn) for _ in range(2))
  v = torch.randn(shape, device="cuda:0", generator=g).mul_(0.3).to(torch.bfloat16)
  scales = dict(q_scale=torch.rand(H, device="cuda:0", generator=g) * 0.2 + 0.1, k_scale=torch.rand(H, device="cuda:0", generator=g) * 0.2 + 0.1)
  table = torch.randn((H, 2 * L - 1), device="cuda:0", generator=g) * 0.05 if pos else None
  outs = []
  for flags in (0, _lib.FWD_COMPILER_SCHEDULED_BLOCKS):
    out = torch.full(v.shape, float("nan"), device=v.device, dtype=v.dtype)
    a, keep = hstu_ops.build_args(q, k, v, out, pos_bias=table, **scales, **kw)
    assert hstu_ops.kernel_variant(a) == "hstu_fwd_mfma_fp8"
    a.flags |= flags
    hstu_ops._run(a, keep)
    torch.cuda.synchronize()
    outs.append(out)
  assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
  b, n = 0, int(lens[0])                         # the longest sequence against the oracle
  pick = (lambda x: x[:n][None]) if jagged else (lambda x: x[b:b + 1, :n])
  qf, kf = (pick(x.float() * s[:, None]).cpu().numpy() for x, s in ((q, scales["q_scale"]), (k, scales["k_scale"])))
  okw = dict(pos_tab=table.cpu().numpy()) if pos else {}
  ref = O.hstu_attention_ref(qf, kf, pick(v).float().cpu().numpy(), n=L, causal=causal, **okw)
  got = pick(outs[0]).float().cpu().numpy()
  assert np.abs(got - ref).max() <= 2e-2 * np.abs(ref).max()
