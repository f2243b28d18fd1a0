"""Callers that were built against earlier versions of the two C ABIs: their structs are prefixes of today's and are taken as they are."""

import ctypes as C

import pytest

from recml_amd import _lib, _lib_block


def _prefix(struct, stop):
  """The struct as it was before the field `stop`."""
  fields = []
  for f in struct._fields_:
    if f[0] == stop:
      break
    fields.append(f)
  return type(struct.__name__ + "Before", (C.Structure,), {"_fields_": fields})


FWD3 = _prefix(_lib.HstuAttnFwdArgs, "mask_pitch")


class BWD3(C.Structure):
  _fields_ = [("fwd", FWD3) if f[0] == "fwd" else f for f in _lib.HstuAttnBwdArgs._fields_]


def _as(struct, source, version=3):
  """`source` in an earlier struct, field by field."""
  a = struct()
  for f in struct._fields_:
    value = getattr(source, f[0])
    setattr(a, f[0], _as(f[1], value, version) if isinstance(value, C.Structure) else value)
  if hasattr(a, "version"):
    a.struct_size, a.version = C.sizeof(struct), version
  return a


def _backward():
  b = _lib.HstuAttnBwdArgs()
  b.struct_size, b.version = C.sizeof(b), _lib.ABI_VERSION
  b.fwd = _lib.new_args()
  f = b.fwd
  f.B, f.L, f.Lkv, f.H, f.d_qk, f.d_v = 2, 256, 256, 4, 64, 64
  f.q = f.k = f.v = f.out = 0x10000
  f.q_stride_t = f.k_stride_t = f.v_stride_t = f.o_stride_t = 4 * 64
  f.q_stride_h = f.k_stride_h = f.v_stride_h = f.o_stride_h = 64
  f.q_stride_b = f.k_stride_b = f.v_stride_b = f.o_stride_b = 256 * 4 * 64
  f.alpha, f.inv_n, f.causal = 1.0, 1.0 / 256, 1
  f.qk_dtype = f.v_dtype = f.out_dtype = _lib.DTYPE_BF16
  f.dropout_p, f.dropout_seed = 0.25, 7          # (the last fields of version 3)
  b.dout = b.dq = b.dk = 0x20000
  b.dv = 0x20004                                 # off a 16-byte boundary: seen only if it is read from where version 3 has it
  return b


def test_attention_takes_version_3():
  lib = _lib.load()
  b = _backward()
  b3 = _as(BWD3, b)
  ptr = lambda x, t: C.cast(C.byref(x), C.POINTER(t))
  fwd = lambda x: ptr(x, _lib.HstuAttnFwdArgs)
  assert lib.hstu_attn_fwd_variant(fwd(b3.fwd)) == lib.hstu_attn_fwd_variant(C.byref(b.fwd)) == b"hstu_fwd_mfma_bf16"
  b3.fwd.mask = b.fwd.mask = 0x50000
  assert lib.hstu_attn_fwd_workspace_bytes(fwd(b3.fwd)) == lib.hstu_attn_fwd_workspace_bytes(C.byref(b.fwd)) > 0
  b3.fwd.mask = b.fwd.mask = None
  bwd = lambda x: ptr(x, _lib.HstuAttnBwdArgs)
  assert lib.hstu_attn_bwd_variant(bwd(b3)) == b"hstu_bwd_general<bf16, bf16 products>"
  b3.dv = 0x20000
  assert lib.hstu_attn_bwd_variant(bwd(b3)) == b"hstu_bwd_mfma_bf16"
  b3.ddense_bias = 0x30000                       # (the struct's last field; validated before any work)
  assert lib.hstu_attn_bwd(bwd(b3), None) == -1 and b"ddense_bias" in lib.hstu_attn_last_error()
  # sizes and versions that do not belong together
  b3.fwd.version = 4
  assert lib.hstu_attn_fwd(fwd(b3.fwd), None) == -2
  b3.fwd.version = 2
  assert lib.hstu_attn_fwd(fwd(b3.fwd), None) == -2
  b.fwd.version = 3
  assert lib.hstu_attn_fwd(C.byref(b.fwd), None) == -2


@pytest.mark.parametrize("name,call,stops", [
    ("HstuNormGateArgs", "hstu_norm_gate_fwd", {3: "seq_offsets", 4: None}),
    ("HstuNormGateBwdArgs", "hstu_norm_gate_bwd", {3: "u_pre", 4: None}),
    ("HstuGemmSiluArgs", "hstu_gemm_silu_fwd", {3: None, 4: None}),
    ("HstuEmbedNormArgs", "hstu_embed_norm_fwd", {3: "row_map", 4: "sums"}),
    ("HstuEmbedGradArgs", "hstu_embed_grad", {4: None}),
    ("HstuGemmArgs", "hstu_gemm", {4: None}),
])
def test_block_steps_take_earlier_versions(name, call, stops):
  lib = _lib_block.load()
  today = getattr(_lib_block, name)
  fn = getattr(lib, call)
  for version in (2, 3, 4, 5, 6):
    struct = _prefix(today, stops[version]) if version in stops else today
    a = struct()
    a.struct_size, a.version = C.sizeof(struct), version
    status = fn(C.cast(C.byref(a), C.POINTER(today)), None)
    assert (status == -2) == (version not in stops and version != _lib_block.ABI_VERSION), (version, status)
  a.struct_size, a.version = C.sizeof(struct) + 8, 4
  assert fn(C.cast(C.byref(a), C.POINTER(today)), None) == -2


@pytest.mark.gpu
def test_a_version_3_call_runs(gpu):
  import torch
  g = torch.Generator().manual_seed(1)
  q, k, v, dout = (torch.randn((2, 256, 4, 64), generator=g).to("cuda:0").to(torch.bfloat16) for _ in range(4))
  lib, lens = _lib.load(), torch.tensor([256, 99], dtype=torch.int32, device="cuda:0")
  outs = []
  for old in (False, True):
    b = _backward()
    out, dq, dk, dv = (torch.zeros_like(q) for _ in range(4))
    f = b.fwd
    f.q, f.k, f.v, f.out, f.seq_lens, f.mask_mode = q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lens.data_ptr(), _lib.MASK_LENGTH
    b.dout, b.dq, b.dk, b.dv = dout.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr()
    assert lib.hstu_attn_fwd_workspace_bytes(C.byref(f)) == 0      # (small enough to go without a work list)
    call = _as(BWD3, b) if old else b
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.hstu_attn_fwd(C.cast(C.byref(call.fwd), C.POINTER(_lib.HstuAttnFwdArgs)), stream) == 0
    assert lib.hstu_attn_bwd(C.cast(C.byref(call), C.POINTER(_lib.HstuAttnBwdArgs)), stream) == 0
    outs.append([out, dq, dk, dv])
  torch.cuda.synchronize()
  assert all(torch.equal(a, b) and a.abs().sum() > 0 for a, b in zip(*outs))
