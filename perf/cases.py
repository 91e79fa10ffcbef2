"""What the speed of this package is measured on: quantized Linears as a diffusion
transformer calls them, from the one-row modulation Linears to the feed-forward layers of a
video model, and the FP8 quantizers for activations that cross GPUs.

Everything goes through the public entry points: `quantize()` converts the Linears once (that
is what a program keeps), `ln_modulate_quant`, `linear_batch`, `linear_on_cat`, the converted
Linears themselves, `fp8_rowwise_quant` + `float8_inference_scaled_mm`, and `comm_quant`.
Attention and the element-wise glue of a block are PyTorch's and not part of a case; their
results (`attn`, `attn_text`) are inputs here.

Kinds of cases
  linear   one converted Linear on one activation
  ffn      Linear + GELU-tanh + Linear
  double   the Linears of a double-stream (joint attention) block
  single   the Linears of a single-stream block with a parallel MLP
  op       per-row quantizer and scaled matmul as two ops (the reference's op boundary)
  comm     quantize / dequantize of what crosses GPUs around an attention
"""
import torch
from torch import nn

import cache_dit_amd as cda
from cache_dit_amd import comm_quant, ops

DEV = "cuda"
BF16 = torch.bfloat16
_OUT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_OUT_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
  return [
      # AdaLN modulation of a FLUX single-stream block at batch 1: one row, 28 MB of weights.
      # Pure latency: launches, the host's path to them, and a weight stream.
      {"name": "modulation_one_row", "kind": "linear", "quant": "float8_per_row", "m": 1, "k": 3072,
       "n": 9216, "gelu": False},
      # The same with classifier-free guidance (two rows) in weight-only mode, double-stream width.
      {"name": "modulation_guidance_w8a16", "kind": "linear", "quant": "float8_weight_only", "m": 2,
       "k": 3072, "n": 18432, "gelu": False},
      # First MLP Linear of the text stream on its own (256 tokens: Qwen-Image's text length), as a
      # model without the stage patch calls it.
      {"name": "text_mlp_256", "kind": "linear", "quant": "float8_per_row", "m": 256, "k": 3072,
       "n": 12288, "gelu": True},
      # Weight-only projection of a short prompt: an odd number of tokens.
      {"name": "text_proj_77_w8a16", "kind": "linear", "quant": "float8_weight_only", "m": 77,
       "k": 4096, "n": 3072, "gelu": False},
      # Widths that are multiples of 16 and of nothing more: all that the conversion policy asks
      # of a Linear. An odd number of tokens as well.
      {"name": "ragged_widths", "kind": "linear", "quant": "float8_per_row", "m": 1357, "k": 2224,
       "n": 4464, "gelu": True},
      # float8_per_tensor (also what the policy falls back to) at FLUX size.
      {"name": "per_tensor_4608", "kind": "linear", "quant": "float8_per_tensor", "m": 4608, "k": 3072,
       "n": 3072, "gelu": False},
      # The scaled matmul behind the reference's op boundary with an fp16 output, odd row count.
      {"name": "scaled_mm_fp16_1021", "kind": "op", "m": 1021, "k": 3072, "n": 3072, "out": "fp16"},
      # The 16 Linears of a FLUX double-stream block, 4096 image and 512 text tokens.
      {"name": "double_block_4096_512", "kind": "double", "image": 4096, "text": 512, "dim": 3072},
      # The 6 Linears of a FLUX single-stream block on all 4608 tokens.
      {"name": "single_block_4608", "kind": "single", "tokens": 4608, "dim": 3072},
      # Weight-only feed-forward at the Qwen-Image token count (odd: 83 x 83 patches).
      {"name": "ffn_6889_w8a16", "kind": "ffn", "quant": "float8_weight_only", "m": 6889, "dim": 3072,
       "inner": 12288},
      # Feed-forward of the Wan2.1-14B-shaped video model: the largest Linears there are.
      {"name": "video_ffn_32760", "kind": "ffn", "quant": "float8_per_row", "m": 32760, "dim": 5120,
       "inner": 13824},
      # q/k/v encoded for the exchange and decoded, the attention output likewise.
      {"name": "comm_4608", "kind": "comm", "tokens": 4608, "heads": 24, "head_dim": 128},
  ]


def _spread(rng, low, high, step=1):
  """A multiple of `step` between `low` and `high`, spread over the logarithm."""
  x = low * (high / low)**rng.random()
  return min(max(step * round(x / step), step * -(-low // step)), step * (high // step))


def _quant(rng):
  return rng.choice(("float8_per_row", "float8_per_row", "float8_weight_only", "float8_per_tensor"))


def draw(rng):
  kind = rng.choice(("rows", "tokens", "tokens", "ragged", "ffn", "op", "double", "single", "comm"))
  if kind == "rows":  # modulation and other conditioning Linears: a batch of embeddings
    return {"kind": "linear", "quant": rng.choice(("float8_per_row", "float8_weight_only")),
            "m": rng.randint(1, 16), "k": _spread(rng, 1024, 5120, 64), "n": _spread(rng, 1024, 18432, 64),
            "gelu": False}
  if kind == "tokens":  # the projections of prompts and of images, model widths
    return {"kind": "linear", "quant": _quant(rng), "m": _spread(rng, 17, 6889),
            "k": _spread(rng, 1024, 15360, 128), "n": _spread(rng, 1024, 12288, 64), "gelu": rng.random() < 0.3}
  if kind == "ragged":  # any width that is converted
    return {"kind": "linear", "quant": _quant(rng), "m": _spread(rng, 17, 2048),
            "k": _spread(rng, 256, 3072, 16), "n": _spread(rng, 256, 4608, 16), "gelu": rng.random() < 0.3}
  if kind == "ffn":
    dim = _spread(rng, 1024, 5120, 128)
    return {"kind": "ffn", "quant": rng.choice(("float8_per_row", "float8_weight_only")),
            "m": _spread(rng, 256, 16384), "dim": dim, "inner": 128 * round(dim * rng.choice((2.7, 4)) / 128)}
  if kind == "op":
    return {"kind": "op", "m": _spread(rng, 17, 6889), "k": _spread(rng, 1024, 12288, 128),
            "n": _spread(rng, 1024, 12288, 64), "out": rng.choice(("bf16", "fp16", "fp32"))}
  if kind == "double":
    return {"kind": "double", "image": _spread(rng, 1024, 6889), "text": _spread(rng, 33, 512),
            "dim": _spread(rng, 1536, 3072, 128)}
  if kind == "single":
    return {"kind": "single", "tokens": _spread(rng, 1024, 6889), "dim": _spread(rng, 1536, 3072, 128)}
  return {"kind": "comm", "tokens": _spread(rng, 512, 8192), "heads": rng.randint(8, 30),
          "head_dim": rng.choice((64, 128))}


# ------------------------------------------------------------------------------ preparation


def _normal(shape, g, std=1.0):
  return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).mul_(std).to(BF16)


def _activation(m, k, g):
  """Rows of N(0, 1) in which 0.1 % of the channels are outliers (x 20)."""
  x = torch.randn((1, m, k), generator=g, device=DEV, dtype=torch.float32)
  x[..., torch.randint(0, k, (max(1, k // 1000), ), generator=g, device=DEV)] *= 20.0
  return x.to(BF16)


def _linears(widths, quant, g, gelu=()):
  """{name: (in, out)} -> converted Linears with weights N(0, 0.02) and biases N(0, 0.01);
  `gelu` names those whose GELU-tanh is folded into the Linear."""
  net = nn.ModuleDict({name: nn.Linear(k, n, device=DEV, dtype=BF16) for name, (k, n) in widths.items()})
  with torch.no_grad():
    for lin in net.values():
      lin.weight.copy_(_normal(lin.weight.shape, g, 0.02))
      lin.bias.copy_(_normal(lin.bias.shape, g, 0.01))
  cda.quantize(net, cda.QuantizeConfig(quant_type=quant))
  for name in gelu:
    cda.fuse_gelu_tanh_(net[name], nn.GELU(approximate="tanh"))
  return net


def prepare(case, seed):
  g = torch.Generator(device=DEV).manual_seed(seed)
  kind = case["kind"]
  s = {"case": case}
  with torch.no_grad():
    if kind == "linear":
      s["net"] = _linears({"proj": (case["k"], case["n"])}, case["quant"], g, ("proj", ) if case["gelu"] else ())
      s["x"] = _activation(case["m"], case["k"], g)
    elif kind == "ffn":
      s["net"] = _linears({"up": (case["dim"], case["inner"]), "down": (case["inner"], case["dim"])},
                          case["quant"], g, ("up", ))
      s["x"] = _activation(case["m"], case["dim"], g)
    elif kind == "op":
      s["x"] = _activation(case["m"], case["k"], g)
      s["w"], s["w_scale"] = ops.fp8_rowwise_quant(_normal((case["n"], case["k"]), g, 0.02))
      s["bias"] = _normal((case["n"], ), g, 0.01)
    elif kind == "double":
      d = case["dim"]
      square = ("to_q", "to_k", "to_v", "add_q", "add_k", "add_v", "to_out", "to_add_out")
      widths = {name: (d, d) for name in square}
      widths.update(norm=(d, 6 * d), norm_context=(d, 6 * d), up=(d, 4 * d), down=(4 * d, d),
                    up_context=(d, 4 * d), down_context=(4 * d, d))
      s["net"] = _linears(widths, "float8_per_row", g, ("up", "up_context"))
      s["temb"] = torch.nn.functional.silu(_normal((1, d), g))
      for name, rows in (("hidden", case["image"]), ("encoder", case["text"]), ("attn", case["image"]),
                         ("attn_text", case["text"]), ("hidden2", case["image"]), ("encoder2", case["text"])):
        s[name] = _activation(rows, d, g)
    elif kind == "single":
      d = case["dim"]
      widths = {"to_q": (d, d), "to_k": (d, d), "to_v": (d, d), "norm": (d, 3 * d), "proj_mlp": (d, 4 * d),
                "proj_out": (5 * d, d)}
      s["net"] = _linears(widths, "float8_per_row", g, ("proj_mlp", ))
      s["temb"] = torch.nn.functional.silu(_normal((1, d), g))
      s["hidden"], s["attn"] = _activation(case["tokens"], d, g), _activation(case["tokens"], d, g)
    else:
      n, d = case["heads"], case["head_dim"]
      s["qkv"] = _normal((1, case["tokens"], 3, n, d), g)
      s["attn"] = _normal((1, case["tokens"], n * d), g)
  return s


# -------------------------------------------------------------------------------- one pass


def _modulation(lin, temb, parts):
  return [t[:, None] for t in lin(temb).chunk(parts, dim=1)]


def run(s):
  kind = s["case"]["kind"]
  with torch.no_grad():
    if kind == "linear":
      return s["net"]["proj"](s["x"])
    if kind == "ffn":
      return s["net"]["down"](s["net"]["up"](s["x"]))
    if kind == "op":
      q, scale = ops.fp8_rowwise_quant(s["x"])
      bias = s["bias"].to(_OUT[s["case"]["out"]])
      out = ops.float8_inference_scaled_mm(q, scale, s["w"].t(), s["w_scale"].t(), _OUT[s["case"]["out"]], bias=bias)
      return {"codes": q, "scale": scale, "out": out}
    if kind == "double":
      net = s["net"]
      shift1, scale1, gate1, shift2, scale2, gate2 = _modulation(net["norm"], s["temb"], 6)
      c_shift1, c_scale1, c_gate1, c_shift2, c_scale2, c_gate2 = _modulation(net["norm_context"], s["temb"], 6)
      normed = cda.ln_modulate_quant(s["hidden"], shift1, scale1)
      c_normed = cda.ln_modulate_quant(s["encoder"], c_shift1, c_scale1)
      (q, k, v), (cq, ck, cv) = cda.linear_batch([(normed, [net["to_q"], net["to_k"], net["to_v"]]),
                                                  (c_normed, [net["add_q"], net["add_k"], net["add_v"]])])
      (o, ), (co, ) = cda.linear_batch([(s["attn"], [net["to_out"]]), (s["attn_text"], [net["to_add_out"]])])
      normed = cda.ln_modulate_quant(s["hidden2"], shift2, scale2)
      c_normed = cda.ln_modulate_quant(s["encoder2"], c_shift2, c_scale2)
      (h, ), (ch, ) = cda.linear_batch([(normed, [net["up"]]), (c_normed, [net["up_context"]])])
      (f, ), (cf, ) = cda.linear_batch([(h, [net["down"]]), (ch, [net["down_context"]])])
      return {"qkv": [q, k, v], "text_qkv": [cq, ck, cv], "out": [o, co], "ff": [f, cf],
              "gates": [gate1, gate2, c_gate1, c_gate2]}
    if kind == "single":
      net = s["net"]
      shift, scale, gate = _modulation(net["norm"], s["temb"], 3)
      normed = cda.ln_modulate_quant(s["hidden"], shift, scale)
      ((mlp, q, k, v), ) = cda.linear_batch([(normed, [net["proj_mlp"], net["to_q"], net["to_k"], net["to_v"]])])
      return {"qkv": [q, k, v], "out": cda.linear_on_cat(net["proj_out"], [s["attn"], mlp]), "gate": gate}
    sent = comm_quant.fp8_comm_qkv_permute_quant(s["qkv"])
    q, k, v = (comm_quant.fp8_comm_qkv_permute_dequant(part) for part in sent)
    sent_out = comm_quant.fp8_comm_per_token_quant(s["attn"])
    return {"sent": sent.view(torch.uint8), "qkv": [q, k, v], "sent_out": sent_out.view(torch.uint8),
            "out": comm_quant.fp8_comm_per_token_dequant(sent_out)}


# ------------------------------------------------------------------- what a pass cannot do without


def work(case):
  kind = case["kind"]

  def weight(k, n):  # codes, scale and bias
    return k * n + 6 * n

  if kind == "linear":
    m, k, n = case["m"], case["k"], case["n"]
    return {"bytes": 2 * m * k + weight(k, n) + 2 * m * n, "flops": 2.0 * m * k * n}
  if kind == "ffn":
    m, d, i = case["m"], case["dim"], case["inner"]
    return {"bytes": 4 * m * d + weight(d, i) + weight(i, d), "flops": 4.0 * m * d * i}
  if kind == "op":
    m, k, n = case["m"], case["k"], case["n"]
    return {"bytes": 3 * m * k + 4 * m + weight(k, n) + _OUT_BYTES[case["out"]] * m * n,
            "flops": 2.0 * m * k * n}
  if kind == "double":
    d, rows = case["dim"], case["image"] + case["text"]
    # per stream: three inputs, q/k/v, two outputs of d columns; 24 d^2 weights with the modulation
    return {"bytes": 2 * rows * d * (3 + 5) + 36 * d * d + 6 * 30 * d + 2 * d + 2 * 12 * d,
            "flops": 2.0 * rows * 12 * d * d + 2.0 * 12 * d * d}
  if kind == "single":
    d, rows = case["dim"], case["tokens"]
    return {"bytes": 2 * rows * d * (2 + 4) + 15 * d * d + 6 * 11 * d + 2 * d + 2 * 3 * d,
            "flops": 2.0 * rows * 12 * d * d + 2.0 * 3 * d * d}
  t, n, d = case["tokens"], case["heads"], case["head_dim"]
  return {"bytes": 2 * (3 * t * n * (2 * d + d + 4) + t * (3 * n * d + 2)), "flops": 0.0}


def tolerance(case):
  """About four times what the present kernels differ by from the same arithmetic in 64 bits
  (identical codes and scales, one rounding to the output's type)."""
  kind = case["kind"]
  if kind == "comm":
    return "exact"  # bytes, and one rounding of a product of two of them
  if kind in ("double", "single") or (kind == "ffn" and case["quant"] != "float8_weight_only"):
    # a bf16 activation computed in another order moves codes (and now and then the maximum,
    # and with it the scale, of a row) of the quantization behind it: up to 1.4e-2 measured
    return {"rel": 3e-2}
  # bf16 1.7e-3, fp16 2.1e-4 (the rounding itself), fp32 about 1e-4 (the matrix core's FP8 sums)
  return {"rel": {"bf16": 6e-3, "fp16": 8e-4, "fp32": 4e-4}[case.get("out", "bf16")]}
