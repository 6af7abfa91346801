"""Performance cases: the work a program has this framework do, through its
public entry points, from the smallest calls to the largest.

The codec's callers are training and serving programs that keep BF16 weights,
saved activations and optimizer state compressed:

* they decode a weight before each use and encode an activation after it
  (``compress``, ``decompress``), from a 257 x 333 matrix of a few codec blocks
  to a 16384 x 8192 one;
* they advance compressed state in place (``LCTTensor.mul_add_``,
  ``add_comp_``, ``mul_add_many``);
* they multiply by compressed weights (``A_compBT``) and train layers whose
  weights and saved activations are compressed (``RMSLinear``,
  ``Relu2Linear``, forward and backward).

A case is a dict of plain values; ``kind`` picks the path and ``data`` what the
tensor holds.  The codec is lossless and deterministic, so everything but the
two cases with matrix products is compared exactly.
"""
from __future__ import annotations

import math

import torch

from losslessly_compressed_tensors_amd.codec.geometry import geometry
from losslessly_compressed_tensors_amd.comp_format import Distribution, DistType, NoiseLevel
from losslessly_compressed_tensors_amd.components.layers import (
    Linear, RMSLinear, Relu2Linear, compress_weight, flush_saved, prefetch_saved,
    prefetch_weights)
from losslessly_compressed_tensors_amd.LCTensor import LCTTensor
from losslessly_compressed_tensors_amd.operations import A_compBT, compress, decompress
from losslessly_compressed_tensors_amd.tensor_buffer import TensorBuffer

# What a tensor holds -> the codebook a program gives it.
#   weight      N(0, 0.02^2), the training integration's weight codebook
#   momentum    N(0, 1e-3^2), its momentum codebook
#   normal      N(0, 1), the headline tensor
#   activation  N(0, 1) with channels of different scale, the activation codebook
#   relu2       post-ReLU activations, half of them exact zeros
#   medium      N(0, 0.02^2) in the wider layout for data with some noise
#   noisy       N(0, 1) with rows 64 times larger, in the widest layout
_BOOKS = {
    "weight": (DistType.LAPLACE, NoiseLevel.CLEAN, 0.01),
    "momentum": (DistType.EMPIRICAL, NoiseLevel.CLEAN, 0.02),
    "normal": (DistType.GAUSSIAN, NoiseLevel.CLEAN, None),
    "activation": (DistType.LAPLACE, NoiseLevel.CLEAN, None),
    "relu2": (DistType.LAPLACE, NoiseLevel.SPARSE, 0.5),
    "medium": (DistType.GAUSSIAN, NoiseLevel.MEDIUM, None),
    "noisy": (DistType.EMPIRICAL, NoiseLevel.HIGH, None),
}
BUFFER_BYTES = 64 * 2 ** 20   # the trainer's shared arena

# The GPT-2-small shape's block width and MLP width, and one layer's worth of
# tokens (8 sequences of 1024).
WIDTH, HIDDEN, TOKENS = 768, 3072, 8192


def _book(data: str) -> Distribution:
    family, level, zero = _BOOKS[data]
    if zero is None:
        return Distribution(family, noise_level=level)
    return Distribution(family, noise_level=level, zero_prob=zero)


def listed() -> list:
    return [
        # Decode before use.  The smallest calls: a few codec blocks of odd
        # size, where a call costs one block's latency and its launch.
        {"name": "decode_257x333", "kind": "decode", "data": "weight", "rows": 257, "cols": 333,
         "buffered": False},
        # One MLP weight of a small model, in the shared arena.
        {"name": "decode_768x3072", "kind": "decode", "data": "weight", "rows": WIDTH,
         "cols": HIDDEN, "buffered": True},
        # One MLP weight of a large model.
        {"name": "decode_4096x11008", "kind": "decode", "data": "weight", "rows": 4096,
         "cols": 11008, "buffered": True},
        # The largest: the headline tensor.
        {"name": "decode_16384x8192", "kind": "decode", "data": "normal", "rows": 16384,
         "cols": 8192, "buffered": False},
        # Encode.  A small weight stored by itself (a checkpoint being
        # compressed tensor by tensor).
        {"name": "compress_768x768", "kind": "compress", "data": "weight", "rows": WIDTH,
         "cols": WIDTH, "buffered": False},
        # The largest, into the shared arena.
        {"name": "compress_16384x8192", "kind": "compress", "data": "normal", "rows": 16384,
         "cols": 8192, "buffered": True},
        # One activation's life: saved compressed in the forward pass, decoded
        # and freed in the backward pass (odd token count).
        {"name": "activation_8191x3072", "kind": "roundtrip", "data": "relu2", "rows": TOKENS - 1,
         "cols": HIDDEN, "buffered": True},
        # Optimizer state and weights advanced in place, compressed throughout:
        # the momentum and the weight of one large MLP matrix.
        {"name": "momentum_4096x11008", "kind": "momentum", "data": "momentum", "rows": 4096,
         "cols": 11008, "buffered": True},
        {"name": "weight_4096x11008", "kind": "step", "data": "weight", "rows": 4096,
         "cols": 11008, "buffered": True},
        # The weights of one shape of a small model's blocks, stepped together.
        {"name": "weights_8x768x768", "kind": "group", "data": "weight", "rows": WIDTH,
         "cols": WIDTH, "count": 8, "buffered": True},
        # Serving: a decode step's few tokens through a compressed weight.
        {"name": "linear_16x4096x11008", "kind": "linear", "data": "weight", "rows": 11008,
         "cols": 4096, "tokens": 16, "buffered": False},
        # Training: a block's MLP forward and backward, weights and saved
        # activations compressed.
        {"name": "mlp_8192x768x3072", "kind": "mlp", "data": "weight", "rows": HIDDEN,
         "cols": WIDTH, "tokens": TOKENS, "buffered": True},
    ]


def _log_uniform(rng, low: float, high: float) -> float:
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _matrix(rng, low: int, high: int) -> tuple:
    """Rows and columns, odd ones among them, of low..high elements."""
    numel = _log_uniform(rng, low, high)
    cols = int(_log_uniform(rng, 64, min(16384, numel / 16)))
    if rng.random() < 0.5:
        cols = max(64, cols // 64 * 64)
    return max(1, int(numel / cols)), cols


def draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "compress", "compress", "roundtrip", "momentum",
                       "step", "group", "linear", "mlp"])
    case = {"kind": kind, "buffered": True}
    if kind in ("decode", "compress", "roundtrip"):
        rows, cols = _matrix(rng, 2 ** 16, 2 ** 26)
        case.update(data=rng.choice(sorted(_BOOKS)), rows=rows, cols=cols,
                    buffered=kind == "roundtrip" or rng.random() < 0.5)
    elif kind in ("momentum", "step"):
        rows, cols = _matrix(rng, 2 ** 16, 4096 * 11008)
        case.update(data="momentum" if kind == "momentum" else "weight", rows=rows, cols=cols,
                    buffered=rng.random() < 0.75)
    elif kind == "group":
        rows, cols = _matrix(rng, 2 ** 16, 2 ** 21)
        case.update(data="weight", rows=rows, cols=cols, count=rng.randint(2, 8))
    elif kind == "linear":
        case.update(data="weight", rows=64 * int(_log_uniform(rng, 8, 172)),
                    cols=64 * int(_log_uniform(rng, 8, 64)),
                    tokens=int(_log_uniform(rng, 1, 512)), buffered=rng.random() < 0.5)
    else:
        width = 64 * rng.randint(4, 16)
        case.update(data="weight", rows=4 * width, cols=width,
                    tokens=int(_log_uniform(rng, 256, 8192)))
    return case


def _generator(seed: int, stream: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(1000003 * stream + seed)


def _normal(shape, seed: int, stream: int, std: float = 1.0) -> torch.Tensor:
    x = torch.randn(shape, generator=_generator(seed, stream), device="cuda")
    return x.mul_(std).to(torch.bfloat16)


def _tensor(data: str, rows: int, cols: int, seed: int, stream: int = 0) -> torch.Tensor:
    if data in ("weight", "medium"):
        return _normal((rows, cols), seed, stream, 0.02)
    if data == "momentum":
        return _normal((rows, cols), seed, stream, 1e-3)
    x = _normal((rows, cols), seed, stream)
    if data == "relu2":
        return x.relu_()
    if data == "activation":
        scale = torch.rand(cols, generator=_generator(seed, stream + 50), device="cuda")
        return x.mul_((0.25 + 1.5 * scale).to(torch.bfloat16))
    if data == "noisy":
        x[::64].mul_(64)
    return x


def _fields(record) -> dict:
    """What a compressed record stores: the payload words, the side bytes, the
    center and its decode table, the overflow counts and per-block list and,
    for a record of its own storage, the overflow entries.  (In a shared arena
    the entries' place depends on what else lives there; the round trip and
    the decodes return what they decode to.)"""
    block_symbols, lanes, _, words = record.codec_geometry
    payload = record.size // block_symbols * lanes * words   # four unwritten words follow
    out = {"payload": record.data[:payload], "side": record.sign_mantissa,
           "center": record.center, "decode_table": record.decode_table,
           "count": record.fallback_count, "used": record.fallback_used,
           "blocks": record.fallback_blocks}
    if record.fallback_descriptor is None:
        out.update(lanes=record.fallback_lanes, starts=record.fallback_starts,
                   tails=record.fallback_buffer)
    return out


def _buffer(case: dict):
    return TensorBuffer(BUFFER_BYTES, device="cuda") if case["buffered"] else None


def _scalar(value: float) -> torch.Tensor:
    return torch.full((1,), value, dtype=torch.float32, device="cuda")


def _mlp_inputs(case: dict, seed: int) -> tuple:
    """x, the output's gradient, the norm gains, and (weight, bias) of the two
    projections."""
    tokens, width, hidden = case["tokens"], case["cols"], case["rows"]
    x = _tensor("activation", tokens, width, seed, 1)
    grad = _normal((tokens, width), seed, 2, 1e-2)
    gains = 1 + 0.1 * torch.randn(width, generator=_generator(seed, 3), device="cuda")
    fc = (_normal((hidden, width), seed, 4, 0.02),
          0.02 * torch.randn(hidden, generator=_generator(seed, 5), device="cuda"))
    proj = (_normal((width, hidden), seed, 6, 0.02),
            0.02 * torch.randn(width, generator=_generator(seed, 7), device="cuda"))
    return x, grad, gains, fc, proj


def prepare(case: dict, seed: int) -> dict:
    kind, data, rows, cols = case["kind"], case["data"], case["rows"], case["cols"]
    state = {"kind": kind, "book": _book(data), "buffer": _buffer(case)}
    if kind == "mlp":
        x, grad, gains, fc, proj = _mlp_inputs(case, seed)
        layers = []
        for weight, bias in (fc, proj):
            layer = Linear(weight.shape[1], weight.shape[0]).to("cuda")
            with torch.no_grad():
                layer.weight.copy_(weight)
                layer.bias.copy_(bias)
            compress_weight(layer, state["buffer"], state["book"])
            layers.append(layer)
        state.update(x=x.requires_grad_(), grad=grad, gains=torch.nn.Parameter(gains),
                     fc=layers[0], proj=layers[1], act=_book("activation"),
                     act_relu=_book("relu2"))
        return state
    if kind == "group":
        state["weights"] = [LCTTensor(_tensor(data, rows, cols, seed, 10 + i), state["buffer"],
                                      state["book"]) for i in range(case["count"])]
        # Orthogonalised updates: entries of about 1 / sqrt(cols).
        state["updates"] = [_normal((rows, cols), seed, 30 + i, cols ** -0.5)
                            for i in range(case["count"])]
        state["decay"], state["neg_lr"] = _scalar(1 - 0.035 * 0.025), _scalar(-0.035)
        return state
    x = _tensor(data, rows, cols, seed)
    if kind in ("compress", "roundtrip"):
        state.update(x=x, held=None)
    elif kind == "decode":
        state["record"] = compress(x, state["book"], buffer=state["buffer"])
    elif kind == "momentum":
        state["momentum"] = LCTTensor(x, state["buffer"], state["book"])
        state["grad"] = _normal((rows, cols), seed, 1, 1e-3)
        state["mu"] = _scalar(0.95)
    elif kind == "step":
        state["weight"] = LCTTensor(x, state["buffer"], state["book"])
        state["momentum"] = LCTTensor(_tensor("momentum", rows, cols, seed, 1), state["buffer"],
                                      _book("momentum"))
        state["neg_lr"] = _scalar(-0.01)
    else:
        state["weight"] = compress(x, state["book"], buffer=state["buffer"])
        state["a"] = _normal((case["tokens"], cols), seed, 1)
    return state


def _run_mlp(state: dict) -> dict:
    x, gains, fc, proj = state["x"], state["gains"], state["fc"], state["proj"]
    leaves = (x, gains, fc.weight, fc.bias, proj.weight, proj.bias)
    for leaf in leaves:
        leaf.grad = None
    weights = [fc.weight, proj.weight]
    prefetch_weights(weights)
    z = RMSLinear.apply(x, fc.weight, gains, fc.bias, state["buffer"], True, state["act"])
    out = Relu2Linear.apply(z, proj.weight, proj.bias, state["buffer"], True, state["act_relu"])
    saved = flush_saved()
    out.register_hook(lambda _: (prefetch_weights(weights), prefetch_saved(saved))[1])
    out.backward(state["grad"])
    return {"out": out.detach(), "grad_x": x.grad, "grad_gains": gains.grad,
            "grad_fc": fc.weight.grad, "grad_fc_bias": fc.bias.grad,
            "grad_proj": proj.weight.grad, "grad_proj_bias": proj.bias.grad}


def run(state: dict):
    kind = state["kind"]
    if kind == "decode":
        return decompress(state["record"])
    if kind == "compress":
        # The program drops the record of the pass before, as it would a value
        # it replaces.
        if state["held"] is not None:
            state["held"].free()
        state["held"] = compress(state["x"], state["book"], buffer=state["buffer"])
        return _fields(state["held"])
    if kind == "roundtrip":
        record = compress(state["x"], state["book"], buffer=state["buffer"])
        dense = decompress(record)
        record.free()
        return dense
    if kind == "momentum":
        state["momentum"].mul_add_(state["mu"], state["grad"])
        return _fields(state["momentum"].x)
    if kind == "step":
        state["weight"].add_comp_(state["momentum"], state["neg_lr"])
        return _fields(state["weight"].x)
    if kind == "group":
        LCTTensor.mul_add_many(state["weights"], state["decay"], state["updates"],
                               state["neg_lr"])
        return [_fields(w.x) for w in state["weights"]]
    if kind == "linear":
        return A_compBT(state["a"], state["weight"])
    return _run_mlp(state)


def _compressed_bytes(data: str, numel: int) -> float:
    """Side bytes and payload words of ``numel`` elements."""
    block_symbols, lanes, _, words = geometry(_book(data))
    return numel * (1 + 4 * lanes * words / block_symbols)


def work(case: dict) -> dict:
    kind, data, numel = case["kind"], case["data"], case["rows"] * case["cols"]
    packed, dense = _compressed_bytes(data, numel), 2 * numel
    if kind in ("decode", "compress"):
        return {"bytes": packed + dense, "flops": 0}
    if kind == "roundtrip":
        return {"bytes": 2 * (packed + dense), "flops": 0}
    if kind == "momentum":
        return {"bytes": 2 * packed + dense, "flops": 0}
    if kind == "step":
        return {"bytes": 2 * packed + _compressed_bytes("momentum", numel), "flops": 0}
    if kind == "group":
        return {"bytes": case["count"] * (2 * packed + dense), "flops": 0}
    tokens = case["tokens"]
    if kind == "linear":
        return {"bytes": packed + 2 * tokens * (case["rows"] + case["cols"]),
                "flops": 2 * tokens * numel}
    # x and the output's gradient in, the output and x's gradient out, both
    # weights in (compressed) and both weights' gradients out; six products.
    return {"bytes": 4 * 2 * tokens * case["cols"] + 2 * packed + 2 * dense,
            "flops": 12 * tokens * numel}


def tolerance(case: dict):
    if case["kind"] == "linear":
        return {"rel": 7e-3, "max": 0.2}
    if case["kind"] == "mlp":
        return {"rel": 2e-2, "max": 0.5}
    return "exact"


def exact(case: dict, seed: int):
    kind, rows, cols = case["kind"], case["rows"], case["cols"]
    if kind in ("decode", "roundtrip"):
        return _tensor(case["data"], rows, cols, seed).double()
    if kind == "linear":
        weight = _tensor(case["data"], rows, cols, seed).double()
        return _normal((case["tokens"], cols), seed, 1).double() @ weight.T
    if kind != "mlp":
        return None   # stored bytes, not computed numbers
    x, grad, gains, fc, proj = _mlp_inputs(case, seed)
    # The layers take their gains and biases in the activations' type.
    leaves = [t.to(torch.bfloat16).double().requires_grad_()
              for t in (x, gains, *fc, *proj)]
    x64, gains64, w1, b1, w2, b2 = leaves
    eps = torch.finfo(torch.bfloat16).eps
    rstd = (x64.square().mean(-1, keepdim=True) + eps).rsqrt()
    z = (x64 * rstd * gains64) @ w1.T + b1
    out = z.relu().square() @ w2.T + b2
    out.backward(grad.double())
    names = ("grad_x", "grad_gains", "grad_fc", "grad_fc_bias", "grad_proj", "grad_proj_bias")
    return {"out": out.detach(), **{n: t.grad for n, t in zip(names, leaves)}}
