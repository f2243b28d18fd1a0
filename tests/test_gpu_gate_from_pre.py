"""The gate of a block taken from its pre-activation in the backward."""

import ctypes as C

import pytest
import torch

from recml_amd import _lib_block

pytestmark = pytest.mark.gpu


def _stream():
  return C.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("rows,width", [(1, 8), (37, 64), (129, 200), (66, 512), (9, 1024), (5, 2048)])
def test_gate_from_its_pre_activation(gpu, rows, width):
  """The same bits without reading the gate as from the gate the projection's product stored (silu of the pre-activation, rounded), its
  gradient then put through the activation by a pass of its own."""
  lib = _lib_block.load()
  g = torch.Generator().manual_seed(rows)
  rn = lambda *s: torch.randn(*s, generator=g).to("cuda:0", torch.bfloat16)
  a, pre, dout, gamma, beta = rn(rows, width), rn(rows, width) * 3, rn(rows, width), rn(width), rn(width)
  pre.view(-1)[::7] *= 20                             # (far into both tails)

  # the activation as the projection's product rounds it: silu of bf16 values, rounded
  def product(x):
    eye = torch.eye(width, device="cuda:0", dtype=torch.bfloat16)
    out, z = torch.empty_like(x), torch.empty_like(x)
    m = _lib_block.HstuGemmArgs(struct_size=C.sizeof(_lib_block.HstuGemmArgs), version=_lib_block.ABI_VERSION, op=_lib_block.GEMM_NN,
                                activation=1, M=rows, N=width, K=width, slabs=1, x=x.data_ptr(), x_stride=width, out=out.data_ptr(),
                                pre=z.data_ptr())
    m.w[0] = eye.data_ptr()
    assert lib.hstu_gemm(C.byref(m), _stream()) == 0
    assert torch.equal(z, x)
    return out

  u = product(pre)
  grads = []
  for gate, z in ((u, None), (torch.full_like(u, float("nan")), pre)):
    da, du, sums = torch.empty_like(a), torch.empty_like(a), torch.empty(2, width, device="cuda:0")
    need = lib.hstu_norm_gate_bwd_workspace_bytes(rows, width)
    buf = torch.empty(max(int(need), 16), dtype=torch.uint8, device="cuda:0")
    n = _lib_block.HstuNormGateBwdArgs(struct_size=C.sizeof(_lib_block.HstuNormGateBwdArgs), version=_lib_block.ABI_VERSION, rows=rows, width=width,
                                       eps=1e-6, a=a.data_ptr(), u=gate.data_ptr(), dout=dout.data_ptr(), a_stride=width, u_stride=width,
                                       dout_stride=width, gamma=gamma.data_ptr(), beta=beta.data_ptr(), da=da.data_ptr(), du=du.data_ptr(),
                                       da_stride=width, du_stride=width, dgamma=sums.data_ptr(), dbeta=sums.data_ptr() + 4 * width,
                                       workspace=buf.data_ptr(), workspace_bytes=buf.numel(), u_pre=z.data_ptr() if z is not None else None,
                                       u_pre_stride=width)
    assert lib.hstu_norm_gate_bwd(C.byref(n), _stream()) == 0
    if z is None:
      assert lib.hstu_silu_bwd(du.data_ptr(), width, pre.data_ptr(), width, rows, width, _stream()) == 0
    grads.append((da, du, sums))
  for x, y in zip(*grads):
    assert torch.equal(x, y)


@pytest.mark.parametrize("rows,width", [(0, 16), (3, 8), (1500, 72), (5000, 512)])
def test_rounded_sums(gpu, rows, width):
  """The parameters' gradients in bf16: the fp32 sums, rounded."""
  lib = _lib_block.load()
  g = torch.Generator().manual_seed(rows)
  rn = lambda *s: torch.randn(*s, generator=g).to("cuda:0", torch.bfloat16)
  a, dout, gamma, beta, da = rn(rows, width), rn(rows, width), rn(width), rn(width), rn(rows, width)
  buf = torch.empty(max(int(lib.hstu_norm_gate_bwd_workspace_bytes(rows, width)), 16), dtype=torch.uint8, device="cuda:0")
  got = []
  for call, dtype in ((lib.hstu_norm_gate_bwd, torch.float32), (lib.hstu_norm_gate_bwd_rounded, torch.bfloat16)):
    sums = torch.full((2, width + 4), 7.0, device="cuda:0", dtype=dtype)
    n = _lib_block.HstuNormGateBwdArgs(struct_size=C.sizeof(_lib_block.HstuNormGateBwdArgs), version=_lib_block.ABI_VERSION, rows=rows, width=width,
                                       eps=1e-6, a=a.data_ptr(), dout=dout.data_ptr(), a_stride=width, dout_stride=width, gamma=gamma.data_ptr(),
                                       beta=beta.data_ptr(), da=da.data_ptr(), da_stride=width, dgamma=sums[0].data_ptr(),
                                       dbeta=sums[1].data_ptr(), workspace=buf.data_ptr(), workspace_bytes=buf.numel())
    assert call(C.byref(n), _stream()) == 0
    got.append(sums)
  assert torch.equal(got[0].to(torch.bfloat16), got[1])
