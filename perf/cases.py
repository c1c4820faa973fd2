"""The work a program hands to this package, as measurable cases: quantized linear layers from a decode step of one
row to a prefill chunk of thousands, one at a time and a decoder layer's seven at once, and whole-tensor quantize /
dequantize.

A case is a dict of plain values:
  kind "linear": one quantized matmul.  m, n, k: rows of x, output and input features; x: dtype of x; bits, block
      (-1 = per channel), zp: the weight; act: dynamic int8 activations; entry: how it is called ("op" =
      torch.ops.xla.quantized_matmul, "int8" = torch.ops.xla.quantized_matmul_int8, "module" = XlaQuantizedLinear).
  kind "layer": the seven linears of a decoder layer (q, k, v, o, gate, up, down) as modules, m rows; hidden, kv and
      inter features; bits, block, zp, act as above; graph: the step is captured once and replayed, as a serving
      loop does.
  kind "qdq": quantize a tensor [rows, cols] of dtype x to q, and dequantize the result to dtype out; axis: the
      channel axis, or -1 for per-tensor parameters.
Sizes are those of this repository's benchmark, tuned table and tests, or generic ones in between.
"""
import math

import torch

import xla_amd.experimental.custom_kernel  # noqa: F401  defines torch.ops.xla.quantized_matmul{,_int8}
import xla_amd.experimental.quantized  # noqa: F401  binds torch.ops.quantized_decomposed for GPU tensors
from xla_amd.experimental.xla_quantized_matmul import XlaQuantizedLinear, prepare_weight
from xla_amd.quantization import quantize_weight_rtn

_DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "i8": torch.int8, "u8": torch.uint8}
_SIZE = {"f32": 4, "bf16": 2, "f16": 2, "i8": 1, "u8": 1}


def _linear(name, m, n, k, x="bf16", bits=8, block=-1, zp=False, act=False, entry="op"):
  c = dict(kind="linear", m=m, n=n, k=k, x=x, bits=bits, block=block, zp=zp, act=act, entry=entry)
  return dict(c, name=name) if name else c


def _layer(name, m, hidden=4096, kv=1024, inter=14336, bits=8, block=-1, zp=False, act=False, graph=False):
  c = dict(kind="layer", m=m, hidden=hidden, kv=kv, inter=inter, bits=bits, block=block, zp=zp, act=act, graph=graph)
  return dict(c, name=name) if name else c


def _qdq(name, rows, cols, x="bf16", q="i8", out="f32", axis=0):
  c = dict(kind="qdq", rows=rows, cols=cols, x=x, q=q, out=out, axis=axis)
  return dict(c, name=name) if name else c


def listed():
  return [
      # a small layer in the default dtype, eager: the cost of a call
      _linear("small_f32", 8, 1024, 1024, x="f32"),
      # a decode step of one sequence, eager: seven short memory-bound calls
      _layer("decode_layer_m1", 1),
      # the same for a batch of 32 sequences in a serving loop that captured its step
      _layer("decode_layer_m32_graph", 32, graph=True),
      # the vocabulary projection that ends a decode step
      _linear("vocab_m4", 4, 128256, 4096, entry="module"),
      # blockwise int4 with zero points, a decode batch
      _linear("int4_block_m16", 16, 4096, 4096, bits=4, block=128, zp=True),
      # the same weights in a prefill chunk
      _linear("int4_block_m2048", 2048, 4096, 4096, bits=4, block=128, zp=True, entry="module"),
      # a ragged mid-sized batch (short prompts, several drafted tokens per sequence) against asymmetric f16 weights
      _linear("batch_m100_f16_zp", 100, 6144, 4096, x="f16", zp=True, entry="module"),
      # weight-only prefill
      _linear("prefill_m2048", 2048, 14336, 4096, entry="module"),
      # W8A8 prefill through the dedicated operator: bf16 in, bf16 out
      _linear("w8a8_m2048", 2048, 14336, 4096, act=True, entry="int8"),
      # a chunk of a chunked prefill, W8A8, all of a decoder layer's linears
      _layer("w8a8_layer_m512", 512, act=True),
      # feature counts that are no multiple of any tile
      _linear("odd_m40", 40, 3000, 2000),
      # a weight through quantize / dequantize per channel
      _qdq("qdq_channel", 14336, 4096),
  ]


def _log(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
  """One more case.  Rows from 1 to 2048, features from the hundreds to the width of a vocabulary, every dtype and
  weight form; a case is cut (in rows, then in features) to the cost of the largest listed one."""
  kind = rng.choice(["linear"] * 7 + ["layer"] * 2 + ["qdq"])
  if kind == "qdq":
    rows, cols = _log(rng, 64, 14336), _log(rng, 64, 14336)
    if rng.random() < 0.7:
      cols = max(64, cols // 64 * 64)
    return _qdq(None, rows, cols, x=rng.choice(["f32", "bf16", "f16"]), q=rng.choice(["i8", "i8", "u8"]),
                out=rng.choice(["f32", "bf16"]), axis=rng.choice([0, 0, 1, -1]))
  weight = rng.choice(["int8", "int8", "int8_zp", "block4_zp", "block4", "block8", "w8a8", "w8a8"])
  bits = 4 if weight.startswith("block4") else 8
  zp, act = weight.endswith("zp"), weight == "w8a8"
  if kind == "layer":
    hidden = rng.choice([1024, 2048, 2560, 4096])
    inter = hidden * rng.choice([3, 4]) - rng.choice([0, 256])
    return _layer(None, _log(rng, 1, 512), hidden=hidden, kv=hidden // rng.choice([1, 4]), inter=inter, bits=bits,
                  block=128 if weight.startswith("block") else -1, zp=zp, act=act, graph=rng.random() < 0.5)
  x = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
  n, k = _log(rng, 256, 32768), 128 * _log(rng, 4, 112)
  block = rng.choice([128, 128, 256]) if weight.startswith("block") else -1
  if block == -1 and not act and rng.random() < 0.1:
    k = _log(rng, 100, 2000)  # no multiple of the kernels' 128-column blocks
    n = min(n, 3000)
    m = _log(rng, 1, 40)
  else:
    n = n if block == -1 and rng.random() < 0.5 else max(256, n // 64 * 64)
    k = k // block * block if block > 0 else k
    # the dearer kinds of arithmetic get fewer rows: f32 products, a rounding sequence per block
    cost = (6 if x == "f32" and not act else 1) * (3 if block > 0 else 1)
    most = int(2048 * 14336 * 4096 / cost / (n * k))
    m = min(_log(rng, 1, 2048), max(1, most))
  return _linear(None, m, n, k, x=x, bits=bits, block=block, zp=zp, act=act, entry=rng.choice(["op", "module"]))


# ---- inputs -----------------------------------------------------------------------------------------------------


def _activations(g, m, k, dtype, outliers):
  x = torch.randn(m, k, generator=g, device="cuda")
  if outliers:  # dynamic activation quantization meets a few channels of large values
    x[:, torch.randperm(k, generator=g, device="cuda")[:max(1, k // 100)]] *= 20.0
  return x.to(dtype)


def _weight(g, n, k, bits, block, zp, act, dtype):
  """(w_int, scaler, zero_point) of a normally distributed weight, in the operator's layouts."""
  w = torch.randn(n, k, generator=g, device="cuda").mul_(0.02)
  return quantize_weight_rtn(w, bits, block, symmetric=not zp, scale_dtype=torch.float32 if act else dtype)


def _module(g, n, k, bits, block, zp, act, dtype):
  with torch.device("meta"):  # (its buffers are replaced at once)
    q = XlaQuantizedLinear(k, n, is_symmetric=not zp, block_size=block, int4_weight=bits == 4, quantize_activation=act)
  q.load_quantized_weight(*_weight(g, n, k, bits, block, zp, act, dtype))
  q.prepare()
  return q


def _layer_shapes(c):
  h, kv, inter = c["hidden"], c["kv"], c["inter"]
  return (("q", h, h), ("k", kv, h), ("v", kv, h), ("o", h, h), ("gate", inter, h), ("up", inter, h), ("down", h, inter))


def prepare(case, seed):
  g = torch.Generator(device="cuda").manual_seed(seed)
  c = case
  if c["kind"] == "qdq":
    x = torch.randn(c["rows"], c["cols"], generator=g, device="cuda").mul_(0.02)
    lo, hi = (-128, 127) if c["q"] == "i8" else (0, 255)
    if c["axis"] == -1:
      scale = float(x.abs().max()) / 127
      zero = 0 if c["q"] == "i8" else 128
    else:
      scale = x.abs().amax(1 - c["axis"]).clamp_(min=1e-6) / 127
      zero = torch.full(scale.shape, 0 if c["q"] == "i8" else 128, dtype=torch.int64, device="cuda")
    return dict(case=c, x=x.to(_DT[c["x"]]), scale=scale, zero=zero, lo=lo, hi=hi)
  form = (c["bits"], c["block"], c["zp"], c["act"])
  if c["kind"] == "layer":
    mods = {name: _module(g, n, k, *form, torch.bfloat16) for name, n, k in _layer_shapes(c)}
    xs = {k: _activations(g, c["m"], k, torch.bfloat16, c["act"]) for k in (c["hidden"], c["inter"])}
    state = dict(case=c, calls=[(mods[name], xs[k]) for name, _, k in _layer_shapes(c)])
    if c["graph"]:
      _step(state)  # (a capture wants a warm program)
      torch.cuda.synchronize()
      state["graph"] = torch.cuda.CUDAGraph()
      with torch.cuda.graph(state["graph"]):
        state["out"] = _step(state)
    return state
  dtype = _DT[c["x"]]
  x = _activations(g, c["m"], c["k"], dtype, c["act"])
  if c["entry"] == "module":
    return dict(case=c, x=x, module=_module(g, c["n"], c["k"], *form, dtype))
  w, s, z = _weight(g, c["n"], c["k"], *form, dtype)
  if not c["act"]:
    prepare_weight(w, c["block"], c["bits"] == 4, dtype)
  return dict(case=c, x=x, w=w, s=s, z=z)


# ---- one pass ---------------------------------------------------------------------------------------------------


@torch.no_grad()
def _step(state):
  return [module(x) for module, x in state["calls"]]


@torch.no_grad()
def run(state):
  c = state["case"]
  if c["kind"] == "layer":
    if not c["graph"]:
      return _step(state)
    state["graph"].replay()
    return state["out"]
  if c["kind"] == "qdq":
    ops = torch.ops.quantized_decomposed
    x, scale, zero, lo, hi, qdt, out = (state["x"], state["scale"], state["zero"], state["lo"], state["hi"], _DT[c["q"]],
                                        _DT[c["out"]])
    if c["axis"] == -1:
      q = ops.quantize_per_tensor(x, scale, zero, lo, hi, qdt)
      return q, ops.dequantize_per_tensor(q, scale, zero, lo, hi, qdt, out_dtype=out)
    q = ops.quantize_per_channel(x, scale, zero, c["axis"], lo, hi, qdt)
    return q, ops.dequantize_per_channel(q, scale, zero, c["axis"], lo, hi, qdt, out_dtype=out)
  if c["entry"] == "module":
    return state["module"](state["x"])
  if c["entry"] == "int8":
    return torch.ops.xla.quantized_matmul_int8(state["x"], state["w"], state["s"], quantize_activation=c["act"])
  return torch.ops.xla.quantized_matmul(state["x"], state["w"], state["s"], state["z"], block_size=c["block"],
                                        int4_weight=c["bits"] == 4, quantize_activation=c["act"])


# ---- what a pass cannot do without ------------------------------------------------------------------------------


def _linear_work(m, n, k, xb, bits, block, zp, act, out_b):
  scales = n * (k // block if block > 0 else 1) * (2 if zp else 1) * (4 if act else xb)
  return n * k * bits // 8 + m * k * xb + scales + m * n * out_b, 2 * m * n * k


def work(case):
  c = case
  if c["kind"] == "qdq":
    e = c["rows"] * c["cols"]
    return {"bytes": e * (_SIZE[c["x"]] + 2 * _SIZE[c["q"]] + _SIZE[c["out"]]), "flops": 4 * e}
  form = (c["bits"], c["block"], c["zp"], c["act"])
  if c["kind"] == "layer":
    each = [_linear_work(c["m"], n, k, 2, *form, 4 if c["act"] else 2) for _, n, k in _layer_shapes(c)]
    return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
  xb = _SIZE[c["x"]]
  out_b = 4 if c["act"] and c["entry"] != "int8" else xb
  b, f = _linear_work(c["m"], c["n"], c["k"], xb, *form, out_b)
  return {"bytes": b, "flops": f}


def tolerance(case):
  """About four times what each path differs by from its own sums done in 64 bits with the same rounding points
  (measured over the listed cases and two dozen drawn ones: rel 9e-5 for bf16, 8e-6 for f16, 4e-7 for f32 results of
  weight-only layers), with room for a small result of which one value rounds to its other neighbour."""
  c = case
  if c["kind"] == "qdq":
    return "exact"  # element by element: one correct answer
  if c["act"]:
    # exact int32 sums; the scale chain in f32 (4e-8), with one rounding to bf16 in the dedicated operator (1e-5)
    return {"rel": 4e-5, "max": 0.03} if c.get("entry") == "int8" else {"rel": 2e-7, "max": 1e-6}
  # the order of the sums decides which of two neighbours a dot product (of a block, or of all of k) rounds to
  rel, most = {"f32": (2e-6, 2e-5), "f16": (1.2e-4, 8e-3), "bf16": (1e-3, 0.06)}[c.get("x", "bf16")]
  # ... and, with a zero point, which one the row's sum of x rounds to, which moves the whole row (3.5e-4 in f16)
  return {"rel": 8 * rel if c["zp"] and c.get("x", "bf16") != "f32" else rel, "max": most}
