"""Calls small enough to take the position table as it is (no preparation launch): up to 512 keys and just past, ragged lengths,
one table and one per head, causal and full, against the oracle."""

import numpy as np
import pytest
import torch

import recml_amd
from oracle import hstu_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [1, 5, 127, 129, 385, 512, 513])
@pytest.mark.parametrize("d,heads,causal", [(32, 1, True), (64, 3, True), (64, 3, False), (128, 3, True)])
def test_small_call_with_a_position_table(gpu, L, d, heads, causal):
  rng = np.random.default_rng(L + d)
  B, H = 3, 3
  lens = np.array([L, (L + 1) // 2, 1], dtype=np.int32)
  q, k, v = (O.round_bf16(rng.standard_normal((B, L, H, d)).astype(np.float32) * 0.3) for _ in range(3))
  table = (rng.standard_normal((heads, 2 * L - 1)) * 0.3).astype(np.float32)
  ref = O.hstu_attention_ref(q, k, v, seq_lens=lens, causal=causal, pos_tab=np.broadcast_to(table, (H, 2 * L - 1)), dtype=np.float32)
  dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")
  bf = lambda x: dev(x).to(torch.bfloat16)
  out = recml_amd.hstu_attention(bf(q), bf(k), bf(v), seq_lens=dev(lens), pos_bias=dev(table), causal=causal)
  err = lambda x: np.abs(x - ref).max() / np.abs(ref).max()
  assert err(out.float().cpu().numpy()) <= 1e-2
  (qj, off), (kj, _), (vj, _) = (O.padded_to_jagged(x, lens) for x in (q, k, v))
  out = recml_amd.hstu_attention(bf(qj), bf(kj), bf(vj), seq_offsets=dev(off.astype(np.int32)), max_len=L, pos_bias=dev(table), causal=causal)
  assert err(O.jagged_to_padded(out.float().cpu().numpy(), off, L)) <= 1e-2
