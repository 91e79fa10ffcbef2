"""A batch of two activations runs as one launch, or as one per activation where that is the
faster form: counted as kernel nodes of a captured graph, at stages where the two forms were
measured at least 8 % apart."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn
DEV = "cuda"

# image rows, text rows, K, widths of the members, launches
W8A8 = [
    (1184, 59, 2816, [2816] * 3, 1),  # 36 us as one launch, 42 as two
    (1480, 36, 2432, [2432] * 3, 1),  # 33, 39
    (2371, 329, 1664, [1664] * 3, 1),  # 29, 37
    (1157, 148, 3072, [3072] * 3, 1),  # 41, 46
    (2818, 341, 2688, [2688], 1),  # 28, 36
    (4096, 512, 3072, [12288], 2),  # 173, 148
]
W8A16 = [
    (1184, 59, 2816, [2816] * 3, 1),  # 62, 72
    (1058, 123, 3072, [3072] * 3, 1),  # 71, 80
    (1297, 144, 2432, [2432] * 3, 1),  # 58, 64
    (4096, 512, 3072, [12288], 2),
]


def _launches(call):
  from cache_dit_amd import _native
  call()  # attributes are set outside the capture
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph(keep_graph=True)
  with torch.cuda.graph(graph):
    call()
  count = ctypes.c_size_t(0)
  # (the HIP runtime that the library is linked to)
  assert _native.load().hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
  return count.value


def _members(M, K, widths):
  weights = [torch.randint(0, 0x40, (n, K), dtype=torch.uint8, device=DEV).view(FP8) for n in widths]
  scales = [torch.ones(n, device=DEV) for n in widths]
  outs = [torch.empty((M, n), dtype=torch.bfloat16, device=DEV) for n in widths]
  return weights, scales, [None] * len(widths), outs, [0] * len(widths)


@pytest.mark.parametrize("image,text,K,widths,launches", W8A8)
def test_w8a8(image, text, K, widths, launches):
  from cache_dit_amd import ops
  acts = [(torch.ones((M, K), device=DEV).to(FP8), torch.ones(M, device=DEV)) + _members(M, K, widths)
          for M in (image, text)]
  assert _launches(lambda: ops.gemm_rowwise_batched_into(acts)) == launches


@pytest.mark.parametrize("image,text,K,widths,launches", W8A16)
def test_w8a16(image, text, K, widths, launches):
  from cache_dit_amd import ops
  acts = [(torch.ones((M, K), dtype=torch.bfloat16, device=DEV), ) + _members(M, K, widths) for M in (image, text)]
  assert _launches(lambda: ops.w8a16_batched_into(acts)) == launches
