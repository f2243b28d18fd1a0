"""How much scratch a backward asks for (a host function of shapes and options: no GPU needed)."""

import ctypes as C

import pytest

from recml_amd import _lib


def backward_args(B, L, H, d, *, tokens=None, pos=False, ts=False, causal=True, window=-1, fp32=False, Lkv=None):
  """A backward call's struct with addresses that nothing reads; `tokens`: jagged, so many in all."""
  b = _lib.HstuAttnBwdArgs()
  b.struct_size, b.version = C.sizeof(_lib.HstuAttnBwdArgs), _lib.ABI_VERSION
  b.fwd = _lib.new_args()
  f, at = b.fwd, 1 << 20
  f.B, f.L, f.Lkv, f.H, f.d_qk, f.d_v = B, L, Lkv or L, H, d, d
  f.qk_dtype = f.v_dtype = f.out_dtype = 0 if fp32 else 1
  f.q = f.k = f.v = f.out = at
  for x in "qkvo":
    setattr(f, f"{x}_stride_t", H * d)
    setattr(f, f"{x}_stride_h", d)
    setattr(f, f"{x}_stride_b", (f.Lkv if x in "kv" else L) * H * d)
  f.alpha, f.inv_n, f.causal, f.window = 1.0, 1.0 / L, int(causal), window
  if tokens is not None:
    f.layout, f.total_tokens, f.seq_offsets = 1, tokens, at
  if pos:
    f.pos_tab, f.pos_heads, b.dpos_tab = at, H, at
  if ts:
    f.ts_tab, f.ts, f.ts_heads, f.ts_num_buckets, f.ts_bucket_size, b.dts_tab = at, at, 1, 128, 0.301, at
    f.ts_stride_b = 0 if tokens is not None else L
  b.dout = b.dq = b.dk = b.dv = at
  return b


def room_for_kept(b):
  """Bytes beyond what the two kernels need that each form dS for themselves."""
  lib = _lib.load()
  least, best = lib.hstu_attn_fwd_workspace_bytes(C.byref(b.fwd)), lib.hstu_attn_bwd_workspace_bytes(C.byref(b))
  assert best >= least
  return best - least


@pytest.mark.parametrize("d,B,L,mean,tables,kept", [
    # lengths of one mean: a batch of power-law lengths holds two to three times the pairs of one of equal lengths
    (64, 64, 2048, 350, "pos", False), (64, 128, 500, 281, "pos", False), (64, 128, 256, 144, "pos", True), (64, 64, 2048, 350, "", False),
    (64, 64, 2048, 350, "ts", True), (64, 64, 2048, 350, "pos ts", True), (64, 128, 2048, 290, "ts", False),
    (32, 64, 2048, 350, "ts", False), (32, 64, 2048, 350, "pos ts", False), (32, 128, 1024, 170, "ts", True), (32, 16, 1024, 1024, "ts", False), (32, 128, 1024, 170, "pos", False),
    (128, 64, 2048, 350, "", True), (128, 64, 2048, 350, "pos ts", True),
    # one long sequence's tile lasts longer than a round of the chip
    (64, 16, 4096, 900, "pos", True), (64, 16, 4096, 900, "pos frozen", False), (64, 16, 4096, 900, "", False), (32, 16, 4096, 900, "pos ts", False),
])
def test_kept_by_the_bytes_that_a_batch_is_likely_to_have(d, B, L, mean, tables, kept):
  b = backward_args(B, L, 8, d, tokens=B * mean, pos="pos" in tables, ts="ts" in tables)
  if "frozen" in tables:
    b.dpos_tab = b.dts_tab = None
  assert (room_for_kept(b) > 0) == kept


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,L,H,window", [(7, 8192, 8, 256), (24, 8192, 8, 256), (2, 4096, 8, 0), (16, 2048, 8, 31), (16, 2048, 8, 32), (16, 2048, 8, 33), (4, 1000, 8, 100)])
def test_a_window_takes_its_band(B, L, H, window, causal, fp32):
  """Blocks that a sliding window leaves have a slot, not all below the diagonal: a long windowed call stays far below the 4 GiB that are the most."""
  size, block = (16, 1024) if fp32 else (32, 2048)
  n, reach = -(-L // size), -(-window // size)
  band = (reach + 1 if causal else 2 * reach + 1) * n * B * H * block
  b = backward_args(B, L, H, 128, causal=causal, window=window, fp32=fp32, pos=not fp32)
  least = _lib.load().hstu_attn_fwd_workspace_bytes(C.byref(b.fwd))
  assert band <= least + room_for_kept(b) <= band + least + 512
  # a window as wide as the triangle or the square needs no more than they do
  whole = room_for_kept(backward_args(1, 512, H, 128, causal=causal, fp32=fp32))
  assert room_for_kept(backward_args(1, 512, H, 128, causal=causal, window=500, fp32=fp32)) == whole > 0


def test_a_window_leaves_the_cached_head_dims_their_band():
  """Heads of 64 and 32 hand dS on while a likely batch's fit the caches: with a window that is its band."""
  for d in (64, 32):
    assert room_for_kept(backward_args(16, 2048, 8, d, tokens=16 * 2048, ts=True)) == 0 or d == 64
    assert room_for_kept(backward_args(32, 2048, 8, d, tokens=32 * 2048, ts=True)) == 0
    assert room_for_kept(backward_args(32, 2048, 8, d, tokens=32 * 2048, ts=True, window=64)) > 0
