"""The FP8 GEMM's kernel with a workgroup per 32 x 32 tile: rows and columns that leave partial tiles, K below
and above the depth of its ring, whole steps and remainders, every output type, against exact
integers and, bit for bit, against the wide kernel it stands in for."""
import pytest
import torch

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn
DEV = "cuda"
SHAPES = [(17, 8), (32, 32), (33, 40), (65, 1000), (300, 264), (40, 8200)]
KS = [16, 112, 128, 144, 256, 384, 512, 640, 656, 1152, 4240]


@pytest.fixture(autouse=True)
def _auto_variant():
  from cache_dit_amd import _native
  _native.set_gemm_variant(-1)
  yield
  _native.set_gemm_variant(-1)


def _codes(shape, low, high, pad, g):
  """Integers as e4m3, rows of a wider matrix whose other bytes are NaN."""
  full = torch.full((shape[0], shape[1] + pad), float("nan"), device=DEV).to(FP8)
  full[:, :shape[1]] = torch.randint(low, high, shape, generator=g, device=DEV).float().to(FP8)
  return full[:, :shape[1]]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,N", SHAPES)
def test_exact_integers(M, N, dtype):
  """Sums below 9 K < 2^24 and power-of-two scales: exact in any order. The output is a window of a
  buffer of sentinels."""
  from cache_dit_amd import _native, ops
  for K in KS:
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a, w = _codes((M, K), -3, 4, 16, g), _codes((N, K), -3, 4, 32, g)
    sa = torch.pow(2.0, torch.randint(-2, 3, (M, ), generator=g, device=DEV).float())
    sw = torch.pow(2.0, torch.randint(-2, 3, (N, ), generator=g, device=DEV).float())
    b = None if dtype == torch.float32 else torch.randint(-8, 9, (N, ), generator=g, device=DEV).to(dtype)
    want = (a.double() @ w.double().t()) * sa.double()[:, None] * sw.double()
    want = (want if b is None else want + b.double()).float().to(dtype)
    for variant in (-1, 26):
      _native.set_gemm_variant(variant)
      full = torch.full((M + 2, N + 8), 777.0, dtype=dtype, device=DEV)
      ops.gemm_rowwise_into(a, sa, w, sw, b, full[1:M + 1, :N], 0)
      torch.cuda.synchronize()
      assert torch.equal(full[1:M + 1, :N], want), (K, variant)
      full[1:M + 1, :N] = 777.0
      assert bool((full == 777.0).all()), (K, variant)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(17, 72, 640), (77, 528, 1024), (300, 264, 2944), (129, 520, 656), (65, 1000, 2224)])
def test_bits_of_the_wide_kernel(M, N, K, dtype):
  from cache_dit_amd import _native, ops
  g = torch.Generator(device=DEV).manual_seed(M + N + K)
  a = torch.randn(M, K, generator=g, device=DEV).to(FP8)
  w = torch.randn(N, K, generator=g, device=DEV).to(FP8)
  sa, sw = torch.rand(M, generator=g, device=DEV), torch.rand(N, generator=g, device=DEV)
  b = None if dtype == torch.float32 else torch.randn(N, generator=g, device=DEV).to(dtype)
  for epilogue in (0, 1):
    outs = []
    for variant in (26, 17, 18):
      _native.set_gemm_variant(variant)
      outs.append(torch.empty(M, N, dtype=dtype, device=DEV))
      ops.gemm_rowwise_into(a, sa, w, sw, b, outs[-1], epilogue)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]), epilogue


@pytest.mark.parametrize("M,N", [(512, 1536), (512, 1568), (640, 2048), (640, 2080)])
@pytest.mark.parametrize("K", [128, 256, 1008, 1024, 1040, 1152])
def test_on_both_sides_of_the_tile_rule(M, N, K):
  """768 and 784 tiles (fp32 outputs, whole steps to K = 1024), 1280 and 1300 (remainders to K = 1024 and one or two steps,
  whose sums are in full fp32 there: products of 448 x 448 that cancel next to products of a few units). Longer K
  has other rules."""
  from cache_dit_amd import _native, ops
  choice = _native.load().cdit_debug_gemm_choice
  assert (choice(0, M, N, 1024, 2) == 26) == (M * N <= 512 * 1536) and (choice(0, M, N, 1008, 2) == 26) == (M * N <= 640 * 2048)
  g = torch.Generator(device=DEV).manual_seed(M + N + K)
  a, w = _codes((M, K), -3, 4, 16, g), _codes((N, K), -3, 4, 16, g)
  one_m, one_n = torch.ones(M, device=DEV), torch.ones(N, device=DEV)
  if K % 128 or (K < 384 and M * N <= 512 * 1536):
    a[:, 5] = a[:, 13] = 448.0
    w[:, 5], w[:, 13] = 448.0, -448.0
  want = (a.double() @ w.double().t()).float()
  for dtype in (torch.float32, torch.bfloat16):
    out = torch.empty(M, N, dtype=dtype, device=DEV)
    ops.gemm_rowwise_into(a, one_m, w, one_n, None, out, 0)
    torch.cuda.synchronize()
    assert torch.equal(out, want.to(dtype)), dtype


@pytest.mark.parametrize("positive", [False, True])
@pytest.mark.parametrize("M,N", [(2, 40), (9, 264), (16, 8)])
def test_few_rows_have_the_16_row_kernels_bits(M, N, positive):
  """Up to 16 rows either kernel may run, and a sum is in four parts on both: same bits for every type, bias and
  epilogue, with no, one, two and three empty parts. fp32 outputs against 64-bit sums: with K remainders a part is a
  chain of fp32 roundings, at most one per 8 products, each of 2^-24 of what is summed by then; for whole steps
  the FP8 instruction drops what is some 13 places below its largest product, from each product at most 2^-13
  of that, in either direction (as often up as down for normal values, all one way for positive ones)."""
  from cache_dit_amd import _native, ops
  for K in (16, 112, 128, 144, 256, 400, 640, 1152, 1296, 5120, 15360, 15376):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a, w = (torch.randn(n, K, generator=g, device=DEV) for n in (M, N))
    a, w = ((t.abs() if positive else t).mul_(100.0).clamp_(-448, 448).to(FP8) for t in (a, w))
    sa, sw = torch.rand(M, generator=g, device=DEV), torch.rand(N, generator=g, device=DEV)
    for dtype in (torch.float32, torch.bfloat16, torch.float16):
      b = None if dtype == torch.float32 else torch.randn(N, generator=g, device=DEV).to(dtype)
      scale = sa * (1e-4 if dtype == torch.float16 else 1.0)  # (within fp16's range)
      for bias in (None, b):
        for epilogue in (0, 1):
          outs = []
          for variant in (50, 26):
            _native.set_gemm_variant(variant)
            outs.append(torch.empty(M, N, dtype=dtype, device=DEV))
            ops.gemm_rowwise_into(a, scale, w, sw, bias, outs[-1], epilogue)
          torch.cuda.synchronize()
          if K % 128 or K >= 384:  # (whole steps shorter than that take the instance for remainders)
            assert torch.equal(outs[0], outs[1]), (K, dtype, bias is None, epilogue)
          if dtype == torch.float32 and epilogue == 0:
            ad, wd = a.double() * sa.double()[:, None], w.double() * sw.double()[:, None]
            err = (outs[1].double() - ad @ wd.t()).abs()
            if K % 128 or K < 384:
              bound = (K / 32 + 8) * 2.0**-24 * (ad.abs() @ wd.abs().t())
            else:
              bound = K * 2.0**-13 * ad.abs().amax(1)[:, None] * wd.abs().amax(1)
            assert bool((err <= bound).all()), K
