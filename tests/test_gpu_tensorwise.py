"""GPU parity of the per-tensor FP8 path (`float8_per_tensor`) through the C ABI:
quantizer codes and scales bit-exact against the oracle, Linear forward within the
GEMM tolerance, hipGraph capture."""
import pytest
import torch
from torch import nn

from oracle import torch_oracle as to

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn


def _dev():
  return torch.device("cuda", 0)


@pytest.mark.parametrize("mode", ["bf16div", "fp32div"])
@pytest.mark.parametrize("M,K", [(1, 16), (7, 200), (64, 3072), (300, 520), (4608, 3072), (33, 15360),
                                 (5, 17)])
def test_quantizer_bit_exact(M, K, mode):
  from cache_dit_amd import ops
  g = torch.Generator().manual_seed(M * 31 + K)
  x = (torch.randn(M, K, generator=g) * (0.1 + (M % 5))).to(torch.bfloat16)
  x[M // 2, K // 3] = 37.0  # one outlier sets the tensor's scale
  q_ref, s_ref = to.quantize_tensorwise(x, mode)
  q, s = ops.fp8_tensorwise_quant(x.to(_dev()), mode)
  torch.cuda.synchronize()
  assert torch.equal(s.cpu(), s_ref)
  assert torch.equal(q.cpu().view(torch.uint8), q_ref.view(torch.uint8))


@pytest.mark.parametrize("mode", ["bf16div", "fp32div"])
def test_quantizer_edge_cases(mode):
  from cache_dit_amd import ops
  # all zeros -> scale 1; strided rows; huge and tiny magnitudes (cold division path)
  z = torch.zeros(9, 64, dtype=torch.bfloat16)
  q, s = ops.fp8_tensorwise_quant(z.to(_dev()), mode)
  assert torch.all(s.cpu() == 1.0) and torch.all(q.cpu().view(torch.uint8) == 0)
  for mag in (1e-30, 1e30):
    g = torch.Generator().manual_seed(2)
    x = (torch.randn(12, 256, generator=g) * mag).to(torch.bfloat16)
    q_ref, s_ref = to.quantize_tensorwise(x, mode)
    q, s = ops.fp8_tensorwise_quant(x.to(_dev()), mode)
    assert torch.equal(s.cpu(), s_ref)
    assert torch.equal(q.cpu().view(torch.uint8), q_ref.view(torch.uint8))
  base = torch.randn(20, 512, generator=torch.Generator().manual_seed(4)).to(torch.bfloat16)
  xs = base.to(_dev())[:, :384]  # row stride 512, K 384
  q_ref, s_ref = to.quantize_tensorwise(base[:, :384].contiguous(), mode)
  q, s = ops.fp8_tensorwise_quant(xs, mode)
  assert torch.equal(s.cpu(), s_ref) and torch.equal(q.cpu().view(torch.uint8), q_ref.view(torch.uint8))


def test_repeated_calls_do_not_keep_the_previous_amax():
  from cache_dit_amd import ops
  big = torch.full((8, 64), 100.0, dtype=torch.bfloat16, device=_dev())
  small = torch.full((8, 64), 0.5, dtype=torch.bfloat16, device=_dev())
  _, s1 = ops.fp8_tensorwise_quant(big)
  _, s2 = ops.fp8_tensorwise_quant(small)
  assert torch.all(s1.cpu() == to.choose_scale_tensorwise(big.cpu()))
  assert torch.all(s2.cpu() == to.choose_scale_tensorwise(small.cpu()))


def _ref_linear(x, lin_w, bias, mode="bf16div"):
  xq, xs = to.quantize_tensorwise(x, mode)
  wq, ws = to.quantize_tensorwise(lin_w, mode)
  return to.scaled_mm_rowwise(xq, xs, wq, ws, bias)


@pytest.mark.parametrize("M,K,N", [(1, 256, 512), (77, 384, 264 + 8), (4096, 3072, 3072)])
def test_linear_forward_matches_oracle(M, K, N):
  import cache_dit_amd
  N = (N // 16) * 16
  torch.manual_seed(M + K)
  lin = nn.Linear(K, N, bias=True).to(torch.bfloat16)
  x = torch.randn(M, K).to(torch.bfloat16)
  ref = _ref_linear(x, lin.weight.detach(), lin.bias.detach()).float()
  m = nn.Sequential(lin).to(_dev())
  cache_dit_amd.quantize(m, cache_dit_amd.QuantizeConfig(quant_type="float8_per_tensor",
                                                         regional_quantize=False))
  assert type(m[0]).__name__ == "Fp8DynamicLinearPerTensor"
  assert torch.all(m[0].weight_scale == m[0].weight_scale[0])
  out = m(x.to(_dev())).float().cpu()
  err = (out - ref).abs().max() / ref.abs().max()
  assert err <= 1e-2, err


def test_forward_under_hip_graph_capture():
  import cache_dit_amd
  torch.manual_seed(0)
  m = nn.Sequential(nn.Linear(512, 1024).to(torch.bfloat16)).to(_dev())
  cache_dit_amd.quantize(m, cache_dit_amd.QuantizeConfig(quant_type="float8_per_tensor",
                                                         regional_quantize=False))
  x = torch.randn(96, 512, device=_dev()).to(torch.bfloat16)
  eager = m(x).clone()
  side = torch.cuda.Stream()
  side.wait_stream(torch.cuda.current_stream())
  with torch.cuda.stream(side):
    m(x)
  torch.cuda.current_stream().wait_stream(side)
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    y = m(x)
  for scale in (1.0, 3.0, 0.25):  # the amax scratch must be re-zeroed on every replay
    x.copy_((torch.randn(96, 512, device=_dev()) * scale).to(torch.bfloat16))
    expect = m(x).clone()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, expect)
  assert eager.shape == y.shape


@pytest.mark.parametrize("M", [1, 7, 8, 9, 64, 65, 513, 2047, 2048, 2049, 4608, 16400])
@pytest.mark.parametrize("K", [8, 520, 4104, 6152])
def test_partial_maxima_by_row_count(M, K):
  """The two-kernel form leaves a partial maximum per eight rows (at most one per CU) in the scale
  vector: row counts around those limits, rows that one or several wavefronts cast, the tensor's maximum in the first, a middle and the last
  row, the same buffers again each time (they hold the previous scale), a NaN and an infinity."""
  from cache_dit_amd import ops
  if M * K > 1 << 24:
    pytest.skip("the row counts are covered by the short rows")
  g = torch.Generator().manual_seed(M + K)
  base = torch.randn(M, K, generator=g).clamp_(-3, 3).to(torch.bfloat16)
  q = torch.empty((M, K), dtype=torch.float8_e4m3fn, device=_dev())
  s = torch.empty((M + 4, ), dtype=torch.float32, device=_dev()).fill_(7.0)
  ws = torch.empty((1, ), dtype=torch.int32, device=_dev())
  for row, peak in ((0, 1000.0), (M // 2, -37.0), (M - 1, 5.0), (M - 1, float("inf")), (0, float("nan")), (M // 2, 4.0)):
    x = base.clone()
    x[row, K - 1] = peak
    ops.quant_tensorwise_into(x.to(_dev()), q, s[:M], ws, 0)
    torch.cuda.synchronize()
    amax = x.abs().amax()
    assert int(ws) == int(amax.view(torch.int16)) & 0x7fff
    if not torch.isfinite(amax):
      assert torch.isnan(s[:M]).all() if torch.isnan(amax) else torch.isinf(s[:M]).all()
      continue
    q_ref, s_ref = to.quantize_tensorwise(x, "bf16div")
    assert torch.equal(s[:M].cpu(), s_ref.reshape(-1).expand(M)) and (s[M:] == 7.0).all()
    assert torch.equal(q.cpu().view(torch.uint8), q_ref.view(torch.uint8))


@pytest.mark.parametrize("M,K", [(63, 64), (64, 64), (65, 64), (130, 1024), (2048, 72), (2049, 512), (4097, 1024),
                                 (8193, 200), (4100, 3080), (2050, 4104), (2100, 6152), (2100, 8200)])
def test_rows_in_flight_together(M, K):
  """Whole and partial groups of 64 rows, one to four rows and more per wavefront of the amax kernel
  (2048 wavefronts), rows of one and several wavefronts of the cast: the outlier that sets the scale
  is in turn in the first, the last and a middle row, in its first and its last element."""
  from cache_dit_amd import ops
  x = torch.randn(M, K, generator=torch.Generator().manual_seed(M + K)).to(torch.bfloat16)
  for row, col in ((0, 0), (M - 1, K - 1), (M // 2 + 1, K - 1), (min(2047, M - 1), 0)):
    y = x.clone()
    y[row, col] = -57.0
    q_ref, s_ref = to.quantize_tensorwise(y, "bf16div")
    q, s = ops.fp8_tensorwise_quant(y.to(_dev()), "bf16div")
    torch.cuda.synchronize()
    assert torch.equal(s.cpu(), s_ref), (row, col)
    assert torch.equal(q.cpu().view(torch.uint8), q_ref.view(torch.uint8)), (row, col)
