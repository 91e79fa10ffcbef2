"""The GEMMs' tiles for problems that one round covers (a workgroup per tile, fed by wavefronts of its own): every tile
at partial rows and columns, K shorter than its ring, odd and even numbers of steps, every output type, bit for bit
against the wide kernel; and which problems take them."""
import ctypes

import pytest
import torch

FP8 = torch.float8_e4m3fn
DEV = "cuda"
TILES = {31: (32, 48), 32: (48, 48), 33: (80, 48), 34: (64, 64), 35: (96, 64), 36: (96, 96), 37: (128, 96),
         38: (32, 32), 39: (48, 32)}
WEIGHT_ONLY = {21: (16, 64), 22: (32, 32), 23: (48, 32), 24: (32, 64), 25: (48, 64), 26: (80, 64), 27: (64, 96), 28: (96, 96),
               29: (96, 128)}


@pytest.fixture(autouse=True)
def _auto_variant():
  from cache_dit_amd import _native
  if not _native.is_built():
    pytest.skip("libcdit_hip.so not built")
  _native.set_gemm_variant(-1)
  yield
  _native.set_gemm_variant(-1)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("variant", sorted(TILES))
def test_bits_of_the_wide_kernel(variant, dtype):
  """The output is a window of a buffer of sentinels; what lies beyond K in the operands' rows is NaN. 384 and 640: K of
  which every tile of the wide kernel (3 to 5 steps ahead) takes one."""
  from cache_dit_amd import _native, ops
  bm, bn = TILES[variant]
  for M, N, K in ((17, 8, 640), (bm, bn, 384), (bm + 1, bn + 8, 768), (3 * bm - 15, 9 * bn - 40, 640),
                  (2 * bm + 16, 17 * bn + 16, 1152)):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a, w = torch.full((M, K + 16), float("nan"), device=DEV).to(FP8), torch.full((N, K + 32), float("nan"), device=DEV).to(FP8)
    a[:, :K] = torch.randn(M, K, generator=g, device=DEV).to(FP8)
    w[:, :K] = torch.randn(N, K, generator=g, device=DEV).to(FP8)
    sa, sw = torch.rand(M, generator=g, device=DEV), torch.rand(N, generator=g, device=DEV)
    for bias in ((False, ) if dtype == torch.float32 else (False, True)):
      b = torch.randn(N, generator=g, device=DEV).to(dtype) if bias else None
      for epilogue in (0, 1):
        outs = []
        for v in (variant, 17 if K >= 640 else 15):
          _native.set_gemm_variant(v)
          outs.append(torch.full((M + 2, N + 8), 777.0, dtype=dtype, device=DEV))
          ops.gemm_rowwise_into(a[:, :K], sa, w[:, :K], sw, b, outs[-1][1:M + 1, :N], epilogue)
        torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[1]), (M, N, K, bias, epilogue)
        outs[0][1:M + 1, :N] = 777.0
        assert bool((outs[0] == 777.0).all()), (M, N, K, bias, epilogue)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(77, 3072, 4096), (200, 2560, 8192), (512, 3072, 3072), (250, 12288, 1152)])
def test_the_choice_and_its_neighbours(M, N, K):
  """By shape, against the wide kernel, on both sides of a round: M rows and as many as need one more."""
  from cache_dit_amd import _native, ops
  tile = TILES[_native.load().cdit_debug_gemm_choice(0, M, N, K, 1)]
  g = torch.Generator(device=DEV).manual_seed(M)
  rows = -(-M // tile[0]) * tile[0] + 1
  a = torch.randn(rows, K, generator=g, device=DEV).to(FP8)
  w = torch.randn(N, K, generator=g, device=DEV).to(FP8)
  sa, sw = torch.rand(rows, generator=g, device=DEV), torch.rand(N, generator=g, device=DEV)
  for m in (M, rows - 1, rows):
    outs = []
    for v in (-1, 17):
      _native.set_gemm_variant(v)
      outs.append(torch.empty(m, N, dtype=torch.bfloat16, device=DEV))
      ops.gemm_rowwise_into(a[:m], sa[:m].clone(), w, sw, None, outs[-1], 0)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]), m


@pytest.mark.parametrize("M,N,K,want", [
    (77, 3072, 4096, 39), (200, 2560, 8192, 33), (512, 3072, 3072, 36), (512, 3072, 12288, 36), (1021, 3072, 3072, 37),
    (512, 12288, 3072, 16), (100, 1024, 3072, 38), (4608, 3072, 3072, 14), (2048, 12288, 3072, 15),
    # up to 16 rows, K remainders and K of one or two steps have other rules
    (16, 3072, 3072, 50), (77, 3072, 4112, 26), (77, 3072, 256, 26)])
def test_tile_of_one_round(M, N, K, want):
  from cache_dit_amd import _native
  lib = _native.load()
  assert lib.cdit_debug_gemm_choice(0, M, N, K, 1) == want
  if want not in (14, 16):  # built for bf16 outputs only
    assert lib.cdit_debug_gemm_choice(0, M, N, K, 0) == want
  assert lib.cdit_debug_gemm_choice(0, M, N, 1024, 2) not in TILES  # short K, fp32 outputs: bound by the stores


@pytest.mark.gpu
@pytest.mark.parametrize("variant", sorted(WEIGHT_ONLY))
def test_weight_only_bits_of_the_wide_kernel(variant):
  """As above; K of whole steps of the ring (128 or 64 elements) and of half ones, with remainders, and shorter than a step. The
  wide kernel takes a K remainder with its masked instances."""
  from cache_dit_amd import _native, ops
  bm, bn = WEIGHT_ONLY[variant]
  for M, N, K in ((17, 16, 640), (bm, bn, 384), (bm + 1, bn + 16, 448), (3 * bm - 15, 9 * bn - 48, 656), (5, 2 * bn, 48),
                  (2 * bm + 16, 17 * bn + 16, 1104)):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.full((M, K + 8), float("nan"), device=DEV, dtype=torch.bfloat16)
    w = torch.full((N, K + 32), float("nan"), device=DEV).to(FP8)
    x[:, :K] = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w[:, :K] = torch.randn(N, K, generator=g, device=DEV).to(FP8)
    sw = torch.rand(N, generator=g, device=DEV)
    for b in (None, torch.randn(N, generator=g, device=DEV).bfloat16()):
      for epilogue in (0, 1):
        outs = []
        for v in (variant, 11):
          _native.set_gemm_variant(v)
          outs.append(torch.full((M + 2, N + 8), 777.0, dtype=torch.bfloat16, device=DEV))
          ops.w8a16_into(x[:, :K], w[:, :K], sw, b, outs[-1][1:M + 1, :N], epilogue)
        torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[1]), (M, N, K, b is None, epilogue)
        outs[0][1:M + 1, :N] = 777.0
        assert bool((outs[0] == 777.0).all()), (M, N, K, b is None, epilogue)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(77, 3072, 4096), (200, 2560, 8192), (512, 3072, 3088), (16, 9216, 3072), (16, 6144, 1040)])
def test_weight_only_choice(M, N, K):
  """By shape, against the kernel for 32 x 32 tiles: the same bits."""
  from cache_dit_amd import _native, ops
  lib = _native.load()
  assert lib.cdit_debug_gemm_choice(1, M, N, K, 1) in WEIGHT_ONLY
  g = torch.Generator(device=DEV).manual_seed(M)
  x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
  w, sw = torch.randn(N, K, generator=g, device=DEV).to(FP8), torch.rand(N, generator=g, device=DEV)
  outs = []
  for v in (-1, 13):
    _native.set_gemm_variant(v)
    outs.append(torch.empty(M, N, dtype=torch.bfloat16, device=DEV))
    ops.w8a16_into(x, w, sw, None, outs[-1], 0)
  torch.cuda.synchronize()
  assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("M,N,K,want", [
    (77, 3072, 4096, 21), (200, 2560, 8192, 25), (17, 3072, 3072, 22), (342, 2752, 12352, 26), (6889, 3072, 12288, 8),
    # up to 16 rows on many columns; K of fewer than five steps has other rules
    (16, 8192, 3072, 22), (16, 9216, 3072, 21), (16, 18432, 5120, 13), (16, 3072, 3072, 50), (1, 9216, 3072, 51), (77, 3072, 256, 13),
    (77, 3080, 4096, 3)])
def test_weight_only_tile_of_one_round(M, N, K, want):
  from cache_dit_amd import _native
  assert _native.load().cdit_debug_gemm_choice(1, M, N, K, 1) == want


class _KernelNode(ctypes.Structure):
  """hipKernelNodeParams."""
  _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint32 * 3),
              ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(77, 3072, 4096), (200, 2560, 8192), (512, 3072, 3072), (97, 8192, 3072), (342, 2752, 12352),
                                   (1579, 352, 12032)])
def test_the_choice_is_what_runs(M, N, K):
  """The workgroups of the one kernel that a call launches are the tiles of the variant that the library names."""
  from cache_dit_amd import _native, ops
  lib = _native.load()
  w, sw = torch.zeros(N, K, device=DEV).to(FP8), torch.ones(N, device=DEV)
  out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
  a, sa = torch.zeros(M, K, device=DEV).to(FP8), torch.ones(M, device=DEV)
  x = torch.zeros(M, K, device=DEV, dtype=torch.bfloat16)
  calls = [(1, WEIGHT_ONLY, lambda: ops.w8a16_into(x, w, sw, None, out, 0))]
  if K % 128 == 0:
    calls.append((0, TILES, lambda: ops.gemm_rowwise_into(a, sa, w, sw, None, out, 0)))
  for weight_only, tiles, call in calls:
    bm, bn = tiles[lib.cdit_debug_gemm_choice(weight_only, M, N, K, 1)]
    call()  # attributes are set outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
      call()
    nodes, count, node = (ctypes.c_void_p * 1)(), ctypes.c_size_t(1), _KernelNode()
    # (the HIP runtime that the library is linked to)
    assert lib.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), nodes, ctypes.byref(count)) == 0 and count.value == 1
    assert lib.hipGraphKernelNodeGetParams(ctypes.c_void_p(nodes[0]), ctypes.byref(node)) == 0
    assert list(node.grid) == [-(-M // bm) * -(-N // bn), 1, 1], (weight_only, bm, bn)
