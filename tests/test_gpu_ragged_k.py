"""K that is a multiple of 16 and of nothing more, through every kernel that takes it: exact
integers (every partial sum is below 2^24, so each order of summation gives the same fp32
value and the comparison is bit for bit), operands that are views of wider rows whose
remaining bytes are NaN (a read beyond K that counted would show), outputs framed by
sentinels."""
import pytest
import torch

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn
DEV = "cuda"

# below one step of 128 (64) elements, on both sides of its multiples, below the prefetch depth,
# and long
KS = [16, 48, 112, 144, 240, 272, 336, 656, 1040, 2224]
SHAPES = [(17, 72), (65, 136), (300, 528), (577, 400)]  # edges of the tiles, ragged rows and columns


@pytest.fixture(autouse=True)
def _auto_variant():
  from cache_dit_amd import _native
  _native.set_gemm_variant(-1)
  yield
  _native.set_gemm_variant(-1)


def _ints(low, high, shape, g):
  return torch.randint(low, high, shape, generator=g, device=DEV).float()


def _framed(values, pad, dtype):
  """`values` [R, K] as a view of rows of K + pad elements, the rest NaN."""
  full = torch.full((values.shape[0], values.shape[1] + pad), float("nan"), device=DEV).to(dtype)
  full[:, :values.shape[1]] = values.to(dtype)
  return full[:, :values.shape[1]]


def _problem(M, N, K, seed, act_dtype):
  g = torch.Generator(device=DEV).manual_seed(seed)
  a, w = _ints(-3, 4, (M, K), g), _ints(-3, 4, (N, K), g)
  sa = torch.pow(2.0, torch.randint(-3, 3, (M, ), generator=g, device=DEV).float())
  sw = torch.pow(2.0, torch.randint(-3, 3, (N, ), generator=g, device=DEV).float())
  b = torch.randint(-8, 9, (N, ), generator=g, device=DEV).to(torch.bfloat16)
  # fp64: the reference itself must not round
  exact = (a.double() @ w.double().t()) * sw.double()[None, :]
  return (_framed(a, 32, act_dtype), _framed(w, 48, FP8), sa, sw, b, exact)


def _check(run, exact, M, N, what):
  full = torch.full((M + 2, N + 8), 777.0, dtype=torch.bfloat16, device=DEV)
  run(full[1:M + 1, :N])
  torch.cuda.synchronize()
  assert torch.equal(full[1:M + 1, :N], exact.float().to(torch.bfloat16)), what
  full[1:M + 1, :N] = 777.0
  assert bool((full == 777.0).all()), ("wrote outside the output", what)


@pytest.mark.parametrize("variant", [-1, 12, 14, 15, 16, 17, 18])
def test_w8a8_tiles(variant):
  from cache_dit_amd import _native, ops
  _native.set_gemm_variant(variant)
  for i, K in enumerate(KS):
    for M, N in SHAPES:
      a, w, sa, sw, b, exact = _problem(M, N, K, 7 * i + M, FP8)
      exact = exact * sa.double()[:, None] + b.double()[None, :]
      _check(lambda out: ops.gemm_rowwise_into(a, sa, w, sw, b, out, 0), exact, M, N, (variant, M, N, K))


@pytest.mark.parametrize("variant", [-1, 7, 8, 9, 10, 11, 12])
def test_w8a16_tiles(variant):
  from cache_dit_amd import _native, ops
  _native.set_gemm_variant(variant)
  for i, K in enumerate(KS):
    for M, N in SHAPES:
      # (72 and 136 columns are multiples of 8 and not of 16: the kernel for any shape)
      a, w, _, sw, b, exact = _problem(M, N, K, 11 * i + M, torch.bfloat16)
      exact = exact + b.double()[None, :]
      _check(lambda out: ops.w8a16_into(a, w, sw, b, out, 0), exact, M, N, (variant, M, N, K))


@pytest.mark.parametrize("M", [1, 2, 16])
def test_few_rows(M):
  from cache_dit_amd import ops
  N = 264
  for i, K in enumerate(KS + [4096 - 16, 4096 + 16]):
    a, w, sa, sw, b, exact = _problem(M, N, K, 13 * i + M, FP8)
    want = exact * sa.double()[:, None] + b.double()[None, :]
    _check(lambda out: ops.gemm_rowwise_into(a, sa, w, sw, b, out, 0), want, M, N, ("w8a8", M, K))
    x, w, _, sw, b, exact = _problem(M, N, K, 13 * i + M, torch.bfloat16)
    _check(lambda out: ops.w8a16_into(x, w, sw, b, out, 0), exact + b.double()[None, :], M, N, ("w8a16", M, K))
    # the whole Linear: rows whose maximum is 7 * 64, so that the scale is 1 and the codes are
    # the integers themselves
    x[:, 0] = 448.0
    exact = (x.double() @ w.float().double().t()) * sw.double()[None, :] + b.double()[None, :]
    q = torch.empty((M, K), dtype=FP8, device=DEV)
    s = torch.empty((M, ), dtype=torch.float32, device=DEV)
    _check(lambda out: ops.linear_w8a8_into(x, w, sw, b, out, q, s, 0, 0), exact, M, N, ("linear", M, K))
    assert torch.equal(q.float(), x.float()) and bool((s == 1.0).all())


@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("variant", [15, 17])
def test_other_output_types(out_dtype, variant):
  from cache_dit_amd import _native, ops
  _native.set_gemm_variant(variant)
  for K in KS:
    M, N = 300, 528
    a, w, sa, sw, _, exact = _problem(M, N, K, K, FP8)
    out = torch.empty((M, N), dtype=out_dtype, device=DEV)
    ops.gemm_rowwise_into(a, sa, w, sw, None, out, 0)
    torch.cuda.synchronize()
    assert torch.equal(out, (exact * sa.double()[:, None]).float().to(out_dtype)), (out_dtype, variant, K)


def _wide_range_problem(M, N, K, seed, act_dtype):
  """Products of 448 x 448 = 200704 next to products of a few units, all integers: in each run of
  128 k, two k where every activation is 448 and the weights are +448 and -448, so the large
  products cancel and the result is the sum of the small ones. At most K / 64 = 64 large products
  of 200704 and 9 K small units: every partial sum in any order is an integer below 2^24, exact in
  fp32. A unit that cuts low bits of a sum next to a large product is off by units."""
  g = torch.Generator(device=DEV).manual_seed(seed)
  a, w = _ints(-3, 4, (M, K), g), _ints(-3, 4, (N, K), g)
  for k in range(0, K - 15, 128):
    first = k + int(torch.randint(0, 8, (1, ), generator=g, device=DEV))
    second = first + 8
    a[:, first] = a[:, second] = 448.0
    w[:, first], w[:, second] = 448.0, -448.0
  assert (2 * ((K + 127) // 128)) * 448**2 + 9 * K < 2**24
  exact = a.double() @ w.double().t()
  return _framed(a, 32, act_dtype), _framed(w, 48, FP8), exact


def _expect(run, exact, dtype, what):
  out = torch.empty(exact.shape, dtype=dtype, device=DEV)
  run(out)
  torch.cuda.synchronize()
  assert torch.equal(out, exact.float().to(dtype)), what


@pytest.mark.parametrize("K", [144, 336, 1040, 2224, 4080])
def test_sums_keep_fp32(K):
  """Every kernel that takes such a K sums in full fp32, as the kernels for any shape do."""
  from cache_dit_amd import _native, ops
  for M in (1, 2, 16, 17, 300):
    N = 264
    a, w, exact = _wide_range_problem(M, N, K, K + M, FP8)
    x = _framed(a.float(), 32, torch.bfloat16)
    one, ones = torch.ones(M, device=DEV), torch.ones(N, device=DEV)
    for dtype, variants in ((torch.bfloat16, (-1, 100, 12, 14, 15, 16, 17, 18)), (torch.float16, (-1, 15, 17, 18)),
                            (torch.float32, (-1, 15, 17, 18))):
      for variant in variants if M > 16 else (-1, 50):
        _native.set_gemm_variant(variant)
        _expect(lambda out: ops.gemm_rowwise_into(a, one, w, ones, None, out, 0), exact, dtype,
                (M, K, dtype, variant))
    for variant in (-1, 100, 7, 8, 9, 10, 11, 12) if M > 16 else (-1, 50):
      _native.set_gemm_variant(variant)
      _expect(lambda out: ops.w8a16_into(x, w, ones, None, out, 0), exact, torch.bfloat16, ("w8a16", M, K, variant))
    _native.set_gemm_variant(-1)
    q = torch.empty((M, K), dtype=FP8, device=DEV)
    s = torch.empty((M, ), dtype=torch.float32, device=DEV)
    _expect(lambda out: ops.linear_w8a8_into(x, w, ones, None, out, q, s, 0, 0), exact, torch.bfloat16,
            ("linear", M, K))
    assert torch.equal(q.float(), x.float()) and bool((s == 1.0).all())


@pytest.mark.parametrize("variant", [0, 3, 7, 8, 9, 10, 11, 12])
@pytest.mark.parametrize("M", [2, 16, 17])
def test_w8a16_tiles_need_whole_columns(variant, M):
  """N a multiple of 8 and not of 16: no tile of the wide kernel may be taken, whatever M is and
  whichever is asked for (a lane of it owns 16 columns)."""
  from cache_dit_amd import _native, ops
  _native.set_gemm_variant(variant)
  for N, K in ((264, 112), (8, 48), (1288, 656)):
    a, w, _, sw, b, exact = _problem(M, N, K, N + K + M, torch.bfloat16)
    _check(lambda out: ops.w8a16_into(a, w, sw, b, out, 0), exact + b.double()[None, :], M, N, (variant, M, N, K))


@pytest.mark.parametrize("M,N,K", [(16, 2560, 320), (16, 2576, 320), (16, 18432, 832), (5, 8192, 1600), (5, 8208, 1600),
                                   (3, 13648, 1360), (3, 13664, 1360), (9, 4552, 112), (9, 4568, 112), (9, 4560, 112)])
def test_w8a16_few_rows_on_both_sides_of_the_tile_rule(M, N, K):
  """Up to 16 rows with a K remainder: the 16-row kernel up to 40960 outputs and where N is not a
  multiple of 16, a wavefront per 32 x 32 tile beyond."""
  from cache_dit_amd import _native, ops
  a, w, _, sw, b, exact = _problem(M, N, K, N + K + M, torch.bfloat16)
  for variant in (-1, 50, 13) if N % 16 == 0 else (-1, 50):
    _native.set_gemm_variant(variant)
    _check(lambda out: ops.w8a16_into(a, w, sw, b, out, 0), exact + b.double()[None, :], M, N, (variant, M, N, K))


def _second_tiles(variant, tiles, M, N):
  bm, bn = tiles[variant]
  return -(-M // bm) * -(-N // bn) > torch.cuda.get_device_properties(0).multi_processor_count


@pytest.mark.parametrize("variant,M,N", [(14, 4700, 4112), (15, 4700, 4112), (16, 2500, 2680), (18, 2100, 2096),
                                         (17, 2100, 1808)])
@pytest.mark.parametrize("K", [48, 240, 656])
def test_w8a8_workgroups_take_a_second_tile(variant, M, N, K):
  """More tiles than CUs: the persistent workgroup goes on to another tile, with K below and above
  the prefetch depth (the next tile's first steps are fetched during this one's last, padded
  ones)."""
  from cache_dit_amd import _native, ops
  assert _second_tiles(variant, {14: (288, 192), 15: (256, 192), 16: (128, 192), 18: (128, 128), 17: (64, 128)}, M, N)
  _native.set_gemm_variant(variant)
  a, w, sa, sw, b, exact = _problem(M, N, K, K + variant, FP8)
  exact *= sa.double()[:, None]
  _check(lambda out: ops.gemm_rowwise_into(a, sa, w, sw, b, out, 0), exact + b.double()[None, :], M, N, (variant, K))
  if variant in (15, 17, 18):
    for dtype in (torch.float16, torch.float32):
      out = torch.empty((M, N), dtype=dtype, device=DEV)
      ops.gemm_rowwise_into(a, sa, w, sw, None, out, 0)
      torch.cuda.synchronize()
      assert torch.equal(out, exact.float().to(dtype)), (dtype, variant, K)


@pytest.mark.parametrize("variant,M,N", [(7, 4700, 4112), (8, 4700, 4112), (9, 4700, 4112), (10, 2500, 2688),
                                         (11, 2100, 2112), (12, 2100, 1808)])
@pytest.mark.parametrize("K", [48, 240, 656])
def test_w8a16_workgroups_take_a_second_tile(variant, M, N, K):
  from cache_dit_amd import _native, ops
  tiles = {7: (256, 256), 8: (256, 192), 9: (192, 256), 10: (128, 192), 11: (128, 128), 12: (128, 64)}
  assert _second_tiles(variant, tiles, M, N)
  _native.set_gemm_variant(variant)
  a, w, _, sw, b, exact = _problem(M, N, K, K + variant, torch.bfloat16)
  _check(lambda out: ops.w8a16_into(a, w, sw, b, out, 0), exact + b.double()[None, :], M, N, (variant, K))


@pytest.mark.parametrize("M,N", [(17, 72), (255, 128), (257, 136), (577, 400), (2100, 4112)])
@pytest.mark.parametrize("K", [16, 112, 240, 272, 656, 2224])
def test_w8a8_tile_of_256_by_128(M, N, K):
  """Edges of the tile, one and two tiles per workgroup (2100 x 4112: 297), K below and above the
  prefetch depth: the exact result, and the bits of the 128 x 128 tile with a GELU epilogue."""
  from cache_dit_amd import _native, ops
  a, w, sa, sw, b, exact = _problem(M, N, K, N + K + M, FP8)
  _native.set_gemm_variant(19)
  _check(lambda out: ops.gemm_rowwise_into(a, sa, w, sw, b, out, 0),
         exact * sa.double()[:, None] + b.double()[None, :], M, N, (M, N, K))
  outs = []
  for variant in (19, 18):
    _native.set_gemm_variant(variant)
    outs.append(torch.empty((M, N), dtype=torch.bfloat16, device=DEV))
    ops.gemm_rowwise_into(a, sa, w, sw, b, outs[-1], 1)
  torch.cuda.synchronize()
  assert torch.equal(outs[0], outs[1]), (M, N, K)
