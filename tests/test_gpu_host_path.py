"""The operators' short way through the Python extension (csrc/host_ext.cpp) against the general
Python code, over the forms of arguments that either takes: same bits, same shapes and strides, same
refusals."""
import pytest
import torch

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn
DEV = "cuda"
PLAIN = ("linear_plain", "w8a16_plain", "scaled_mm_plain", "quant_plain", "cat2_plain", "ln_modulate_quant",
         "comm_per_token_quant", "comm_per_token_dequant", "comm_qkv_permute_quant", "comm_qkv_permute_dequant")


class _General:
  """The extension with every function that looks at arguments refusing them."""

  def __init__(self, host):
    self._host = host

  def __getattr__(self, name):
    return (lambda *a: None) if name in PLAIN else getattr(self._host, name)


class _Recorded:
  """The extension, noting for each function that looks at arguments whether it took them."""

  def __init__(self, host):
    self._host, self.taken = host, []

  def __getattr__(self, name):
    f = getattr(self._host, name)

    def call(*a):
      r = f(*a)
      self.taken.append(r is not None)
      return r

    return call if name in PLAIN else f


def _both(monkeypatch, call, plain, skip=0):
  """plain: whether the short way takes the arguments. The first `skip` results are not compared."""
  from cache_dit_amd import _native
  host = _native.host()
  recorded = _Recorded(host)
  with monkeypatch.context() as m:
    m.setattr(_native, "host", lambda: recorded)
    short = call()
    m.setattr(_native, "host", lambda: _General(host))
    general = call()
  # (an op that concatenates and calls another one has that one look as well)
  assert recorded.taken and recorded.taken[0] == plain, recorded.taken
  flat = lambda r: list(r)[skip:] if isinstance(r, (tuple, list)) else [r]  # noqa: E731
  torch.cuda.synchronize()
  assert len(flat(short)) == len(flat(general))
  for a, b in zip(flat(short), flat(general)):
    assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride()
    assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))
  return short


def _forms(K, g):
  """Activations [..., K]: one row, a vector, rows of a wider matrix, more dimensions, dimensions that
  do not merge, columns that are not contiguous."""
  x = torch.randn(6, 20, 2 * K, generator=g, device=DEV).bfloat16()
  return [x[0, :1, :K].contiguous(), x[0, 0, :K].contiguous(), x[0, :, :K], x[:, :, :K].contiguous(), x[1:2, :, :K],
          x[:, ::2, :K], x[0, :, ::2], x.transpose(0, 1)[..., :K]]


@pytest.mark.parametrize("K,N", [(64, 48), (272, 528)])
def test_linears(monkeypatch, K, N):
  from cache_dit_amd import ops
  g = torch.Generator(device=DEV).manual_seed(K)
  w, ws = ops.fp8_rowwise_quant(torch.randn(N, K, generator=g, device=DEV).bfloat16())
  wide = torch.zeros(N, 2 * K, device=DEV).to(FP8)
  wide[:, :K].view(torch.uint8).copy_(w.view(torch.uint8))
  bias = torch.randn(2 * N, generator=g, device=DEV).bfloat16()
  for i, x in enumerate(_forms(K, g)):
    for weight in (w, wide[:, :K]):
      for b in (None, bias[:N], bias[::2]):
        for granularity in (0, 1):
          _both(monkeypatch, lambda: ops.linear_w8a8_op(x, weight, ws, b, i & 1, i & 1, granularity, False),
                i < 4 and (b is None or b.is_contiguous()))
        _both(monkeypatch, lambda: ops.w8a16_mm_op(x, weight.t(), ws, b, 1, i & 1),
              i < 4 and (b is None or b.is_contiguous()))
    q, s = _both(monkeypatch, lambda: ops.fp8_rowwise_quant(x), i < 4)
    for dt, b, plain in ((torch.float16, bias[:N].half(), True), (torch.bfloat16, bias[::2], False),
                         (torch.float32, None, True), (torch.float32, bias[:N].float(), False)):
      _both(monkeypatch, lambda: ops.float8_inference_scaled_mm(q, s, w.t(), ws.t(), dt, bias=b), plain)
    _both(monkeypatch, lambda: ops.float8_inference_scaled_mm(q, s[..., :1].reshape(-1)[:1], w.t().contiguous(), ws[:1],
                                                              torch.bfloat16), False)
    if x.dim() > 1 and K % 16 == 0:
      half = K // 2
      _both(monkeypatch, lambda: ops.linear_w8a8_cat2_op(x[..., :half], x[..., half:], w, ws, bias[:N], 0, 0), i == 2)
      _both(monkeypatch, lambda: ops.linear_w8a8_cat2_op(x[..., :half].contiguous(), x[..., half:].contiguous(), w, ws,
                                                         None, 1, 1), x.numel() // K > 16)


def test_ln_modulate_and_comm(monkeypatch):
  from cache_dit_amd import comm_quant, ops
  K = 64
  g = torch.Generator(device=DEV).manual_seed(1)
  for i, x in enumerate(_forms(K, g)):
    one = torch.randn(2, K, generator=g, device=DEV).bfloat16()
    for write_y in (True, False):  # (an unwritten y is not compared)
      _both(monkeypatch, lambda: ops._ln_modulate_quant_op(x, one[0], one[1], 1e-6, 0, write_y), i < 4, 1 - write_y)
    if x.dim() == 3:
      each = torch.randn(x.shape[0], 1, 2 * K, generator=g, device=DEV).bfloat16()
      _both(monkeypatch, lambda: ops._ln_modulate_quant_op(x, each[..., :K], each[..., K:], 1e-5, 1, True),
            i == 3 and each[..., :K].is_contiguous())
      shift, scale = each[..., :K].contiguous(), each[..., K:].contiguous()
      _both(monkeypatch, lambda: ops._ln_modulate_quant_op(x, shift, scale, 1e-5, 1, True), i == 3)
    packed = _both(monkeypatch, lambda: comm_quant.fp8_comm_per_token_quant(x), x.is_contiguous())
    _both(monkeypatch, lambda: comm_quant.fp8_comm_per_token_dequant(packed), True)
  qkv = torch.randn(2, 9, 3, 4, K, generator=g, device=DEV).bfloat16()
  for x in (qkv, qkv[:, ::2], qkv.transpose(3, 4).contiguous().transpose(3, 4)):
    sent = _both(monkeypatch, lambda: comm_quant.fp8_comm_qkv_permute_quant(x), x.stride(4) == 1)
    for part in (sent[1], sent.transpose(1, 2)[0]):
      _both(monkeypatch, lambda: comm_quant.fp8_comm_qkv_permute_dequant(part), True)


@pytest.mark.parametrize("quant", ["float8_per_row", "float8_weight_only"])
def test_linear_batch(quant):
  """Activations of one to three dimensions, contiguous and not, against the Linears one by one."""
  import cache_dit_amd as cda
  K = 64
  g = torch.Generator(device=DEV).manual_seed(2)
  net = torch.nn.ModuleDict({str(n): torch.nn.Linear(K, n, device=DEV, dtype=torch.bfloat16) for n in (48, 80, 528)})
  cda.quantize(net, cda.QuantizeConfig(quant_type=quant))
  lins = list(net.values())
  forms = _forms(K, g)
  with torch.no_grad():
    for x, other in zip(forms, forms[1:] + forms[:1]):
      single = [[lin(x) for lin in lins[:2]], [lins[2](other)]]
      batch = cda.linear_batch([(x, lins[:2]), (other, lins[2:])])
      for one, many in zip(single, batch):
        for a, b in zip(one, many):
          assert a.shape == b.shape and a.dtype == b.dtype and b.is_contiguous()
          assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def test_empty_and_refused(monkeypatch):
  """No rows; and what was refused stays refused, with the general code's errors."""
  from cache_dit_amd import ops
  K, N = 64, 48
  w = torch.zeros(N, K, device=DEV).to(FP8)
  ws = torch.ones(N, 1, device=DEV)
  x = torch.ones(3, K, device=DEV, dtype=torch.bfloat16)
  none = x[:0]
  _both(monkeypatch, lambda: ops.linear_w8a8_op(none, w, ws, None, 0, 0, 0, False), False)
  _both(monkeypatch, lambda: ops.w8a16_mm_op(none, w.t(), ws, None, 1, 0), False)
  _both(monkeypatch, lambda: ops.fp8_rowwise_quant(none), False)
  for args, match in (((x.float(), w, ws, None, 0, 0, 0, False), "bfloat16"),
                      ((x[:, :48], w, ws, None, 0, 0, 0, False), "shape mismatch"),
                      ((x, w, ws[:5], None, 0, 0, 0, False), "weight_scale"),
                      ((x, w, ws, torch.zeros(N, device=DEV), 0, 0, 0, False), "bias"),
                      ((x, w, ws, None, 2, 0, 0, False), "scale_mode"), ((x, w, ws, None, 0, 0, 2, False), "granularity")):
    with pytest.raises(ValueError, match=match):
      ops.linear_w8a8_op(*args)
  with pytest.raises(ValueError, match="float8_e4m3fn"):
    ops.w8a16_mm_op(x, w.t().float(), ws, None, 1, 0)
  with pytest.raises(ValueError, match="share K"):
    ops.quant_rowwise_batched_into([(x, x.to(FP8), ws[:3, 0])] * 1 + [(x[:, :48], x[:, :48].to(FP8), ws[:3, 0])], 0)
  with pytest.raises(RuntimeError, match="epilogue"):
    ops.linear_w8a8_op(x, w, ws, None, 0, 8, 0, False)
