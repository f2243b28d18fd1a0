"""The block's own matrix products around their tiles, stages, slabs and splits, and the sums of a gathered table's gradient
around their runs, against fp32 products and exact sums."""

import ctypes as C

import pytest
import torch

from recml_amd import _lib_block
from recml_amd import hstu_block_ops as ops

pytestmark = pytest.mark.gpu


def _normal(g, *shape):
  return torch.randn(shape, generator=g).to(torch.bfloat16).to("cuda:0")


def _close(got, want):
  want = want.cpu()
  assert (got.float().cpu() - want).abs().max() <= 8e-3 * want.abs().max().clamp(min=1e-3)


@pytest.mark.parametrize("M,N,K,slabs", [
    (1, 8, 8, 1),              # one piece of one tile
    (65, 72, 40, 1),           # a row past a tile of 64, a contraction that is no whole stage
    (300, 32, 16, 4),          # slabs narrower than a stage: the weight along the contraction is one matrix then
    (257, 160, 136, 4),        # slabs of 40: a stage that crosses from one into the next
    (1000, 512, 128, 4),       # slabs of whole tiles
    (6200, 1024, 136, 2),      # 128 x 128 tiles
    (33000, 512, 1024, 4),     # 256 x 128 tiles of a weight's gradient, a long contraction, a last split that is short
    (6300, 2048, 520, 1),      # 256 x 256 tiles, the last of both axes short; a stage that the contraction ends in
    (6300, 2048, 512, 4),      # the same over slabs
    (9000, 2056, 1032, 1),     # a weight's gradient in four splits, whose 45 tiles two XCDs each share
    (4100, 2056, 2056, 1),     # and in two
])
def test_block_products(gpu, M, N, K, slabs):
  g = torch.Generator().manual_seed(M + N)
  x, y, bias, res = _normal(g, M, K), _normal(g, M, N), _normal(g, N), _normal(g, M, N)
  x = torch.cat([x, x], 1)[:, :K]                                     # rows further apart than they are long
  ws = [_normal(g, K, N // slabs) * 0.1 for _ in range(slabs)]
  w = torch.cat(ws, 1).float()
  want = x.float() @ w + res.float() + bias.float()
  out, pre = ops.block_gemm(_lib_block.GEMM_NN, x, ws, bias=bias, residual=res, activation=True, want_pre=True)
  _close(pre, want)
  _close(out, torch.nn.functional.silu(pre.float()))
  _close(ops.block_gemm(_lib_block.GEMM_NN, x, ws), x.float() @ w)
  if slabs == 1 or N // slabs >= 32:
    _close(ops.block_gemm(_lib_block.GEMM_NT, y, ws), y.float() @ w.t())
  grads = [torch.full_like(t, float("nan")) for t in ws]
  ops.block_gemm(_lib_block.GEMM_TN, x, grads, y=y)
  _close(torch.cat(grads, 1), x.float().t() @ y.float())


@pytest.mark.parametrize("M,N,K", [(16384, 1024, 8), (16400, 1024, 64), (16395, 1032, 64), (1025, 20000, 64), (40000, 480, 200)])
def test_large_outputs(gpu, M, N, K):
  """On either side of the lines of store_past (2^24 outputs; rows of whole 64-byte sectors): the same bits as the products of parts of the
  rows, which are stored the other way and summed in the same order."""
  g = torch.Generator(device="cuda").manual_seed(M + N)
  x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
  w = (torch.randn(K, N, device="cuda", generator=g) * 0.1).to(torch.bfloat16)
  got = ops.gemm_silu(x, w, None, False)
  for at in (slice(0, 700), slice(M - 300, M)):
    assert torch.equal(got[at], ops.gemm_silu(x[at].contiguous(), w, None, False))
  assert bool(torch.isfinite(got).all())


@pytest.mark.parametrize("M,N,K,slabs", [
    (12289, 2048, 512, 4),     # tiles of one row at the end; runs that cross tiles, pieces that cross slabs' ends
    (12288, 2048, 256, 1),     # whole tiles, six pieces for each workgroup
    (36705, 704, 512, 2),      # an odd number of pieces in a tile, slabs of 352: their ends within a piece
    (20000, 1280, 256, 4),
])
def test_rows_in_registers(gpu, M, N, K, slabs):
  """Large products whose rows stay in registers: the same bits as those of parts of the rows, which go by tiles and are summed in the same
  order; and against fp32."""
  g = torch.Generator(device="cuda").manual_seed(M + N)
  x = torch.randn(M, K + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :K]
  ws = [(torch.randn(K, N // slabs, device="cuda", generator=g) * K**-0.5).to(torch.bfloat16) for _ in range(slabs)]
  added = torch.randn(M, N + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :N]
  for kw in ({}, dict(residual=added), dict(activation=True), dict(activation=True, want_pre=True)):
    parts = lambda r: r if isinstance(r, tuple) else (r,)
    got = parts(ops.block_gemm(_lib_block.GEMM_NN, x, ws, **kw))
    for at in range(0, M, 4000):
      part = slice(at, min(at + 4000, M))
      of_part = {k: v[part] if k == "residual" else v for k, v in kw.items()}
      for a, b in zip(got, parts(ops.block_gemm(_lib_block.GEMM_NN, x[part], ws, **of_part))):
        assert torch.equal(a[part], b)
  want = x[-300:].float() @ torch.cat(ws, 1).float()
  _close(got[1][-300:], want)
  _close(got[0][-300:], torch.nn.functional.silu(got[1][-300:].float()))


@pytest.mark.parametrize("M,N,K", [
    (49153, 512, 512),         # a tile of one row at the end; runs that cross tiles
    (49152, 256, 512),         # whole tiles, six pieces for each workgroup
    (36705, 512, 704),         # an odd number of pieces in a tile
])
def test_rows_in_registers_gradient(gpu, M, N, K):
  """Large input gradients, whose weights lie along the contraction: the same bits as those of parts of the rows; and against fp32."""
  g = torch.Generator(device="cuda").manual_seed(M + N)
  d = torch.randn(M, N + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :N]
  w = (torch.randn(K, N, device="cuda", generator=g) * N**-0.5).to(torch.bfloat16)
  got = ops.block_gemm(_lib_block.GEMM_NT, d, [w])
  for at in range(0, M, 4000):
    part = slice(at, min(at + 4000, M))
    assert torch.equal(got[part], ops.block_gemm(_lib_block.GEMM_NT, d[part], [w]))
  _close(got[-300:], d[-300:].float() @ w.float().t())


@pytest.mark.parametrize("M,N,K", [
    (1600, 20000, 64),         # a last tile of 32 columns; every second row begins in the middle of a line
    (900, 20000, 32),
    (1025, 16384, 64),         # a step of one row; whole tiles
    (1, 131080, 128),          # one row, a tile of eight columns
    (256, 16392, 128),         # rows that are no whole sectors
    (1023, 32776, 64),         # the same, wider, and a step without its last row
    (2050, 16416, 128),        # a step of two rows
])
def test_short_contractions(gpu, M, N, K):
  """Large products of a short contraction: the same bits as those of parts of the weight's columns, which go by tiles and are summed in
  the same order; and against fp32."""
  g = torch.Generator(device="cuda").manual_seed(M + N)
  x = torch.randn(M, K + 8, device="cuda", generator=g).to(torch.bfloat16)[:, :K]
  w = (torch.randn(K, N, device="cuda", generator=g) * K**-0.5).to(torch.bfloat16)
  got = ops.block_gemm(_lib_block.GEMM_NN, x, [w])
  for rows in (slice(0, 1000), slice(max(M - 1000, 0), M)):
    for cols in (slice(0, 1024), slice(max(N - 1000, 0), N)):
      assert torch.equal(got[rows, cols], ops.block_gemm(_lib_block.GEMM_NN, x[rows], [w[:, cols].contiguous()]))
  _close(got, x.float() @ w.float())


@pytest.mark.parametrize("M,N,K,slabs", [(32513, 2048, 512, 4), (65281, 1024, 256, 1), (58500, 1152, 512, 2)])
def test_norm_and_product(gpu, M, N, K, slabs):
  """The layer norm and the product as one launch, with tiles of one row at the end and runs that cross tiles, beside the two launches and
  64 bits.  The two round the same values at the same places, but their sums go in other orders: a normed value in some thousands
  falls on the other side of a rounding, 2^-8 of itself, so the errors are alike and few results differ."""
  lib = _lib_block.load()
  assert lib.hstu_norm_gemm_takes(M, N, K, slabs) == 1
  g = torch.Generator(device="cuda").manual_seed(M)
  x = (torch.randn(M, K + 8, device="cuda", generator=g) * 3 + 1).to(torch.bfloat16)[:, :K]
  gamma, beta = ((torch.randn(K, device="cuda", generator=g) * 0.2 + i).to(torch.bfloat16) for i in (1, 0))
  ws = [(torch.randn(K, N // slabs, device="cuda", generator=g) * K**-0.5).to(torch.bfloat16) for _ in range(slabs)]
  out = torch.full((M, N), float("nan"), device="cuda", dtype=torch.bfloat16)
  a = _lib_block.HstuNormGemmArgs()
  a.struct_size, a.version = C.sizeof(a), _lib_block.ABI_VERSION
  a.M, a.N, a.K, a.slabs, a.eps = M, N, K, slabs, 1e-6
  a.x, a.x_stride, a.gamma, a.beta, a.out = x.data_ptr(), x.stride(0), gamma.data_ptr(), beta.data_ptr(), out.data_ptr()
  for i, w in enumerate(ws):
    a.w[i] = w.data_ptr()
  assert lib.hstu_norm_gemm(C.byref(a), C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
  two = ops.block_gemm(_lib_block.GEMM_NN, ops.layer_norm(x.contiguous(), gamma, beta, 1e-6), ws, activation=True)
  xd = x.double()
  xd = (xd - xd.mean(1, keepdim=True)) * torch.rsqrt(xd.var(1, unbiased=False, keepdim=True) + 1e-6)
  want = torch.nn.functional.silu((xd * gamma.double() + beta.double()) @ torch.cat(ws, 1).double())
  err = [float((t.double() - want).norm() / want.norm()) for t in (out, two)]
  assert err[0] <= 1.001 * err[1]
  assert float((out != two).double().mean()) <= 1e-3
  assert float((out.float() - two.float()).abs().max()) <= 2.0**-7 * float(two.float().abs().max())


def test_norm_and_product_sizes(gpu):
  takes = _lib_block.load().hstu_norm_gemm_takes
  assert takes(78000, 2048, 512, 4) == 1 and takes(100000, 1024, 256, 4) == 1
  assert not any([takes(13000, 2048, 512, 4), takes(78000, 2048, 384, 4), takes(78000, 2080, 512, 1), takes(0, 2048, 512, 4),
                  takes(78000, 2048, 512, 5), takes(1 << 31, 2048, 512, 4)])


@pytest.mark.parametrize("rows,keys,width", [(0, 5, 8), (1, 1, 8), (700, 1, 136), (3000, 40, 64), (3000, 5000, 72), (4097, 257, 128)])
@pytest.mark.parametrize("scale", [1.0, 2.0])
def test_gathered_table_gradient(gpu, rows, keys, width, scale):
  """Small whole numbers: every partial sum is exact, whatever is rounded when."""
  g = torch.Generator().manual_seed(rows + keys)
  ids = torch.exp(torch.rand(rows, generator=g).double() * torch.log(torch.tensor(float(keys)))).long() - 1
  ids = ids.clamp(0, keys - 1)
  grad = torch.randint(0, 2, (rows, width), generator=g) * 2 - 1
  grad[torch.rand(rows, generator=g) < 0.7] = 0
  want = torch.zeros(keys, width, dtype=torch.long).index_add_(0, ids, grad) * int(scale)
  assert want.abs().max() < 256
  dev = torch.device("cuda:0")
  d, idd = grad.to(torch.bfloat16).to(dev), ids.to(dev)
  out = torch.full((keys, width), float("nan"), dtype=torch.bfloat16, device=dev)
  lib = _lib_block.load()
  ws = torch.empty(lib.hstu_embed_grad_workspace_bytes(rows, keys, width) + 256, dtype=torch.uint8, device=dev)
  a = _lib_block.HstuEmbedGradArgs()
  a.struct_size, a.version = C.sizeof(a), _lib_block.ABI_VERSION
  a.rows, a.keys, a.width, a.scale = rows, keys, width, scale
  a.g, a.g_stride, a.ids, a.out = d.data_ptr(), width, idd.data_ptr(), out.data_ptr()
  a.workspace = (ws.data_ptr() + 255) // 256 * 256
  a.workspace_bytes = ws.numel() - (a.workspace - ws.data_ptr())
  assert lib.hstu_embed_grad(C.byref(a), C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
  torch.cuda.synchronize()
  assert torch.equal(out.cpu().long(), want)


@pytest.mark.parametrize("width", [72, 136, 512])
@pytest.mark.parametrize("scale", [1.0, 1.7])
def test_long_runs_in_the_order_of_their_tokens(gpu, width, scale):
  """Runs around the batches that are loaded together: every partial sum rounded to bf16, in the tokens' order, bit by bit."""
  lens = [33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 321, 1000]
  g = torch.Generator().manual_seed(width)
  ids = torch.cat([torch.full((n,), k) for k, n in enumerate(lens)])
  ids = ids[torch.randperm(len(ids), generator=g)]
  grad = torch.randn(len(ids), width, generator=g).to(torch.bfloat16)
  want = torch.zeros(len(lens), width, dtype=torch.bfloat16)
  for t, k in enumerate(ids.tolist()):
    want[k] = (want[k].float() + (grad[t].float() * scale).to(torch.bfloat16).float()).to(torch.bfloat16)
  dev = torch.device("cuda:0")
  d, idd, out = grad.to(dev), ids.to(dev), torch.full((len(lens), width), float("nan"), dtype=torch.bfloat16, device=dev)
  lib = _lib_block.load()
  ws = torch.empty(lib.hstu_embed_grad_workspace_bytes(len(ids), len(lens), width) + 256, dtype=torch.uint8, device=dev)
  a = _lib_block.HstuEmbedGradArgs()
  a.struct_size, a.version = C.sizeof(a), _lib_block.ABI_VERSION
  a.rows, a.keys, a.width, a.scale = len(ids), len(lens), width, scale
  a.g, a.g_stride, a.ids, a.out = d.data_ptr(), width, idd.data_ptr(), out.data_ptr()
  a.workspace = (ws.data_ptr() + 255) // 256 * 256
  a.workspace_bytes = ws.numel() - (a.workspace - ws.data_ptr())
  assert lib.hstu_embed_grad(C.byref(a), C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
  torch.cuda.synchronize()
  assert torch.equal(out.cpu(), want)


@pytest.mark.parametrize("B,L,keys,width,by_position", [(128, 9, 9, 72, 2), (192, 3, 5, 136, 2), (20, 40, 40, 128, 2), (128, 9, 9, 64, 1), (30, 7, 9, 136, 1)])
@pytest.mark.parametrize("packed", [False, True])
def test_position_table_gradient(gpu, B, L, keys, width, by_position, packed):
  """The keys are positions, of every entry or of those a row map names.  by_position 2: an fp32 sum rounded once, so at most half a unit
  in the last of its 8 bits off (and what B additions in fp32 leave); by_position 1: exact on whole numbers below 256."""
  g = torch.Generator().manual_seed(B + L)
  rows = torch.arange(B * L) if not packed else (torch.rand(B * L, generator=g) < 0.6).nonzero().squeeze(1)
  T, dev = rows.numel(), torch.device("cuda:0")
  grad = torch.randn((T, width), generator=g).to(torch.bfloat16) if by_position == 2 else torch.randint(-1, 2, (T, width), generator=g).to(torch.bfloat16)
  want = torch.zeros(keys, width, dtype=torch.float64).index_add_(0, rows % L, grad.double())
  d, rm = grad.to(dev), rows.to(torch.int32).to(dev)
  out = torch.full((keys, width), float("nan"), dtype=torch.bfloat16, device=dev)
  lib = _lib_block.load()
  ws = torch.empty(lib.hstu_embed_grad_workspace_bytes(T, keys, width) + 256, dtype=torch.uint8, device=dev)
  a = _lib_block.HstuEmbedGradArgs()
  a.struct_size, a.version = C.sizeof(a), _lib_block.ABI_VERSION
  a.rows, a.keys, a.width, a.scale = T, keys, width, 1.0
  a.g, a.g_stride, a.out, a.L, a.by_position = d.data_ptr(), width, out.data_ptr(), L, by_position
  if packed:
    a.row_map = rm.data_ptr()
  a.workspace = (ws.data_ptr() + 255) // 256 * 256
  a.workspace_bytes = ws.numel() - (a.workspace - ws.data_ptr())
  assert lib.hstu_embed_grad(C.byref(a), C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
  got = out.cpu().double()
  if by_position == 2:
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + B * 2.0 ** -21).all()
  else:
    assert want.abs().max() < 256 and torch.equal(got, want)


@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (5, 8, 7), (64, 20, 12), (65, 17, 65), (130, 40, 100)])
@pytest.mark.parametrize("act", [False, True])
def test_products_of_widths_that_are_no_multiple_of_8(gpu, M, K, N, act):
  """Element by element, fp32 sums and one rounding: 2^-8 of the result, and 2^-20 of the terms' magnitudes for the sums' order."""
  g = torch.Generator().manual_seed(M + N)
  wide = torch.full((M, (K + 15) // 8 * 8), float("nan"), dtype=torch.bfloat16, device="cuda:0")
  wide[:, :K] = _normal(g, M, K)
  x, w, bias = wide[:, :K], _normal(g, K, N), _normal(g, N)
  res = torch.full((M, (N + 15) // 8 * 8), float("nan"), dtype=torch.bfloat16, device="cuda:0")
  res[:, :N] = _normal(g, M, N)
  res = res[:, :N]
  for b, r in ((None, None), (bias, None), (bias, res)):
    want = x.double() @ w.double() + (0 if b is None else b.double()) + (0 if r is None else r.double())
    size = x.double().abs() @ w.double().abs() + 2
    want = torch.nn.functional.silu(want) if act else want
    got = ops.gemm_silu(x, w, b, act, residual=r).double()
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20 * size).all()
