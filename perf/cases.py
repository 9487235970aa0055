"""The work whose speed counts: cases over the range of sizes, data types and directions that users of the TT-NN surface run.

Every case goes through the public entry points (``ttnn``, ``tt_lib``) as model code does: weights are block-float tensors
that stay on the device, activations are in TILE layout, outputs are the tensors that the next op would take.  ``listed()``
names one case for each kind of use; ``draw(rng)`` gives another case of the same ranges.

A case is a dict of plain values.  ``kind`` says which path it takes:

  linear      ttnn.linear(x, w, bias, activation): one projection, decode (few rows) to prefill (thousands)
  mlp         h -> 4h with GELU -> h, the two falcon_* matmuls of a Falcon decoder layer
  gated_mlp   ttnn.linear(silu), ttnn.linear, ttnn.mul, ttnn.linear: the MLP of a Mistral decoder layer
  ffn         ttnn.linear(bias, gelu) with a BFLOAT8_B output, which the second ttnn.linear takes as its activations
  attention   q . k^T and probabilities . v, every head with its own operands
  bmm         activations and block-float operands of their own for every batch slice
  from_torch  a weight matrix in host memory becomes block-float tiles on the device
  to_torch    block-float tiles on the device become an fp32 tensor in host memory
"""
from __future__ import annotations

import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "tt-metal_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import tt_lib  # noqa: E402
import ttnn  # noqa: E402

_DTYPE = {"bf16": ttnn.bfloat16, "bfp8_b": ttnn.bfloat8_b, "bfp4_b": ttnn.bfloat4_b}
_ELEMENT_BYTES = {"fp32": 4.0, "bf16": 2.0, "bfp8_b": 1088 / 1024, "bfp4_b": 576 / 1024}


def listed():
    return [
        # one attention output projection of a decode step for 32 users: the smallest call, launch latency counts
        {"name": "decode_projection", "kind": "linear", "batch": 1, "m": 32, "k": 4096, "n": 4096, "weights": "bfp8_b", "bias": False, "activation": "none"},
        # the MLP of a Falcon-7B decoder layer, decode for 32 users: the ordinary decode step, bound by reading the weights
        {"name": "decode_mlp", "kind": "mlp", "m": 32, "k": 4544, "n": 18176, "weights": "bfp8_b"},
        # the gated MLP of a Mistral-7B decoder layer, decode for 32 users, 4-bit weights
        {"name": "decode_gated_mlp", "kind": "gated_mlp", "m": 32, "k": 4096, "n": 14336, "weights": "bfp4_b"},
        # a decode batch that is no multiple of anything (75 users), Falcon's fused qkv projection
        {"name": "decode_75_users", "kind": "linear", "batch": 1, "m": 75, "k": 4544, "n": 4672, "weights": "bfp8_b", "bias": False, "activation": "none"},
        # a short prompt through the gate projection of the gated MLP
        {"name": "prompt_200", "kind": "linear", "batch": 1, "m": 200, "k": 4096, "n": 14336, "weights": "bfp8_b", "bias": False, "activation": "silu"},
        # a prompt of 1000 tokens (padded to 1024 rows) through the down projection, 4-bit weights
        {"name": "prompt_1000", "kind": "linear", "batch": 1, "m": 1000, "k": 14336, "n": 4096, "weights": "bfp4_b", "bias": False, "activation": "none"},
        # a long prompt through the largest matrix: bound by the matrix cores
        {"name": "prefill_2048", "kind": "linear", "batch": 1, "m": 2048, "k": 4544, "n": 18176, "weights": "bfp8_b", "bias": False, "activation": "none"},
        # the feed-forward block of a BERT-Large encoder layer, batch 8, biases, block-float activations in between
        {"name": "encoder_ffn", "kind": "ffn", "batch": 8, "m": 384, "k": 1024, "n": 4096, "weights": "bfp8_b"},
        # the two batched products of BERT-Large's self-attention, 8 x 16 heads, bf16 operands on both sides
        {"name": "encoder_attention", "kind": "attention", "batch": 8, "m": 384, "k": 64, "weights": "bf16"},
        # a batched product with block-float operands of their own for each of 12 slices
        {"name": "bmm_12", "kind": "bmm", "batch": 12, "m": 384, "k": 1024, "n": 1024, "weights": "bfp8_b"},
        # loading one fp32 weight matrix of a checkpoint from host memory
        {"name": "load_weights", "kind": "from_torch", "batch": 1, "k": 4544, "n": 4672, "source": "fp32", "weights": "bfp8_b"},
        # bringing block-float results of an odd size back to host memory
        {"name": "read_back", "kind": "to_torch", "batch": 1, "k": 1000, "n": 4544, "weights": "bfp8_b"},
    ]


def _spread(rng, low, high):
    """A whole number whose logarithm is spread evenly over [low, high]."""
    return max(low, min(high, round(low * (high / low) ** rng.random())))


def _width(rng, low, high):
    """A matrix extent: mostly whole tiles, as model configurations have them, one in four of any size."""
    extent = _spread(rng, low, high)
    return extent if rng.random() < 0.25 else max(32, (extent + 16) // 32 * 32)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "mlp", "gated_mlp", "ffn", "attention", "bmm", "from_torch", "to_torch"])
    weights = rng.choice(["bfp8_b", "bfp4_b"])
    if kind == "linear":
        return {"kind": kind, "batch": 1, "m": _spread(rng, 1, 2048), "k": _width(rng, 1024, 16384), "n": _width(rng, 1024, 16384) if rng.random() < 0.5 else _width(rng, 1024, 4608),
                "weights": weights, "bias": rng.random() < 0.25, "activation": rng.choice(["none", "none", "gelu", "silu", "relu"])}
    if kind in ("mlp", "gated_mlp"):
        return {"kind": kind, "m": _spread(rng, 1, 512), "k": _width(rng, 1024, 4608), "n": _width(rng, 2816, 16384), "weights": weights}
    if kind == "ffn":
        return {"kind": kind, "batch": rng.randint(1, 8), "m": _spread(rng, 32, 512), "k": _width(rng, 768, 1280), "n": _width(rng, 3072, 5120), "weights": "bfp8_b"}
    if kind == "attention":
        return {"kind": kind, "batch": rng.randint(1, 8), "m": _spread(rng, 64, 512), "k": rng.choice([64, 64, 128]), "weights": rng.choice(["bf16", "bf16", "bfp8_b"])}
    if kind == "bmm":
        return {"kind": kind, "batch": rng.randint(2, 16), "m": _spread(rng, 32, 512), "k": _width(rng, 256, 2048), "n": _width(rng, 256, 2048), "weights": weights}
    if kind == "from_torch":
        return {"kind": kind, "batch": 1, "k": _width(rng, 1024, 4544), "n": _width(rng, 1024, 4672), "source": rng.choice(["fp32", "bf16"]), "weights": weights}
    return {"kind": kind, "batch": 1, "k": _spread(rng, 32, 2048), "n": _width(rng, 1024, 8192), "weights": weights}


_HEADS = 16                                        # of the attention cases (BERT-Large)


def _gemms(case):
    """(batch, m, k, n, weight slices, bytes per weight) of the products of one pass."""
    bytes_per_weight = _ELEMENT_BYTES[case["weights"]]
    m, k, n = case["m"], case["k"], case.get("n")
    if case["kind"] == "attention":
        b = case["batch"] * _HEADS
        return [(b, m, k, m, b, bytes_per_weight), (b, m, m, k, b, bytes_per_weight)]
    if case["kind"] == "mlp":
        return [(1, m, k, n, 1, bytes_per_weight), (1, m, n, k, 1, bytes_per_weight)]
    if case["kind"] == "gated_mlp":
        return [(1, m, k, n, 1, bytes_per_weight)] * 2 + [(1, m, n, k, 1, bytes_per_weight)]
    if case["kind"] == "ffn":
        return [(case["batch"], m, k, n, 1, bytes_per_weight), (case["batch"], m, n, k, 1, bytes_per_weight)]
    return [(case["batch"], m, k, n, case["batch"] if case["kind"] == "bmm" else 1, bytes_per_weight)]


def work(case):
    """Operations of the products, each weight read once, the inputs of the pass read once and its outputs written once
    (bf16); what one op of a pass hands to the next is not counted."""
    if case["kind"] in ("from_torch", "to_torch"):
        dense = _ELEMENT_BYTES[case.get("source", "fp32")]
        return {"bytes": case["batch"] * case["k"] * case["n"] * (dense + _ELEMENT_BYTES[case["weights"]]), "flops": 0}
    gemms = _gemms(case)
    weights = sum(slices * k * n * each for _, _, k, n, slices, each in gemms)
    ends = gemms if case["kind"] == "attention" else [gemms[0], gemms[-1]]
    first = sum(2 * b * m * k for b, m, k, _, _, _ in (ends if case["kind"] == "attention" else ends[:1]))
    last = sum(2 * b * m * n for b, m, _, n, _, _ in (ends if case["kind"] == "attention" else ends[-1:]))
    return {"bytes": weights + first + last, "flops": sum(2 * b * m * k * n for b, m, k, n, _, _ in gemms)}


def tolerance(case):
    if case["kind"] in ("from_torch", "to_torch"):
        return "exact"                             # codes are whole numbers, unpacking is exact
    # Products of exact bf16 operands summed in fp32 and rounded to bf16.  Measured against the same products in 64 bits over the
    # listed cases and drawn ones: 1.7e-3 (the largest difference 3.9e-3, half a step of bf16) where one op writes the output,
    # 1.7e-3 / 5.2e-3 for ffn, 2.4e-3 / 9.6e-3 for mlp and 3.3e-3 / 1.3e-2 for gated_mlp, whose intermediates are rounded
    # too.  Four times that.
    return {"mlp": {"rel": 1e-2, "max": 4e-2}, "gated_mlp": {"rel": 1.3e-2, "max": 5.2e-2}}.get(case["kind"], {"rel": 7e-3, "max": 2.1e-2})


def _normal(generator, shape, scale=1.0):
    return torch.randn(shape, generator=generator, device="cuda", dtype=torch.float32) * scale


def _on_device(tensor, dtype, device):
    """A block-float tensor, or bf16 tiles, as a model's loading code makes them."""
    tensor = tensor.bfloat16() if dtype == ttnn.bfloat16 else tensor
    return ttnn.from_torch(tensor, dtype=dtype, layout=ttnn.TILE_LAYOUT, device=device)


def _inputs(case, seed):
    """The values of one pass as plain tensors, from the seed alone: what a block-float tensor is made from in fp32, the rest in
    the type the path takes."""
    generator = torch.Generator(device="cuda")
    generator.manual_seed(seed)
    kind = case["kind"]

    def activations(*shape):
        return _normal(generator, shape).bfloat16()

    def weights(*shape, scale=0.02):
        return _normal(generator, shape, scale)

    if kind == "from_torch":
        source = weights(case["batch"], 1, case["k"], case["n"])
        return {"host": source if case["source"] == "fp32" else source.bfloat16()}
    if kind == "to_torch":
        return {"x": weights(case["batch"], 1, case["k"], case["n"], scale=1.0)}
    if kind == "attention":
        b, m, d = case["batch"], case["m"], case["k"]
        values = {"q": activations(b, _HEADS, m, d), "k_t": weights(b, _HEADS, d, m, scale=1.0)}
        values["p"] = torch.softmax(_normal(generator, (b, _HEADS, m, m)), dim=-1).bfloat16()
        values["v"] = weights(b, _HEADS, m, d, scale=1.0)
        return values
    b, m, k, n = case.get("batch", 1), case["m"], case["k"], case["n"]
    values = {"x": activations(b, 1, m, k)}
    if kind == "linear":
        values["w"] = weights(1, 1, k, n)
        if case["bias"]:
            values["bias"] = _normal(generator, (1, 1, 1, n), 0.1).bfloat16()
    elif kind == "bmm":
        values["w"] = weights(b, 1, k, n)
    elif kind == "ffn":
        values["w1"], values["w2"] = weights(1, 1, k, n), weights(1, 1, n, k)
        values["b1"], values["b2"] = (_normal(generator, (1, 1, 1, width), 0.1).bfloat16() for width in (n, k))
    elif kind == "mlp":
        values["w1"], values["w2"] = weights(1, 1, k, n), weights(1, 1, n, k)
    else:
        values["w1"], values["w3"], values["w2"] = weights(1, 1, k, n), weights(1, 1, k, n), weights(1, 1, n, k)
    return values


_WEIGHTS = ("k_t", "v", "w", "w1", "w2", "w3")


def prepare(case, seed):
    device = ttnn.open_device(torch.cuda.current_device())
    dtype, kind = _DTYPE[case["weights"]], case["kind"]
    values, state = _inputs(case, seed), {"kind": kind}
    if kind == "from_torch":
        state["host"], state["dtype"], state["device"] = values["host"].cpu(), dtype, device
        return state
    for name, value in values.items():
        state[name] = _on_device(value, dtype if name in _WEIGHTS or kind == "to_torch" else ttnn.bfloat16, device)
    if kind == "linear":
        state.setdefault("bias", None)
        state["activation"] = None if case["activation"] == "none" else case["activation"]
    return state


def _whole_tiles(x):
    return torch.nn.functional.pad(x, (0, -x.shape[-1] % 32, 0, -x.shape[-2] % 32))


def _tiles(x):
    """The elements in the order of 32 x 32 tiles of four 16 x 16 faces, flat."""
    x = _whole_tiles(x)
    h, w = x.shape[-2:]
    return x.reshape(-1, h // 32, 2, 16, w // 32, 2, 16).permute(0, 1, 4, 2, 5, 3, 6).reshape(-1)


def _stored(x, weights):
    """What a tensor of this type holds of x, in 64 bits: for block floats 16 neighbours share the largest one's exponent, and a
    mantissa of 7 or 3 bits is rounded half up."""
    if weights == "bf16":
        return x.bfloat16().double()
    bits = 7 if weights == "bfp8_b" else 3
    groups = _whole_tiles(x).double()
    shape = groups.shape
    groups = groups.reshape(-1, 16)
    step = torch.exp2(torch.frexp(groups.abs().amax(dim=1, keepdim=True))[1].double() - bits)
    codes = torch.clamp(torch.floor(groups.abs() / step + 0.5), max=2 ** bits - 1)
    return (torch.sign(groups) * codes * step).reshape(shape)


def exact(case, seed):
    kind, weights = case["kind"], case["weights"]
    if kind == "from_torch":
        return None
    values = _inputs(case, seed)
    if kind == "to_torch":
        return _stored(values["x"], weights)[..., :case["k"], :case["n"]].cpu()
    values = {name: _stored(value, weights) if name in _WEIGHTS else value.double() for name, value in values.items()}
    # activations are stored in whole tiles: the rows and columns that fill them up are zeros, and part of the outputs
    values = {name: value if name.startswith("b") else _whole_tiles(value) for name, value in values.items()}
    act = {"none": lambda t: t, "gelu": torch.nn.functional.gelu, "silu": torch.nn.functional.silu, "relu": torch.relu}
    pad_bias = lambda t: torch.nn.functional.pad(t, (0, -t.shape[-1] % 32))
    x = values.get("x")
    if kind == "attention":
        return _tiles(values["q"] @ values["k_t"]), _tiles(values["p"] @ values["v"])
    if kind == "linear":
        product = x @ values["w"]
        return _tiles(act[case["activation"]](product + pad_bias(values["bias"]) if case["bias"] else product))
    if kind == "bmm":
        return _tiles(x @ values["w"])
    if kind == "mlp":
        return _tiles(act["gelu"](x @ values["w1"]) @ values["w2"])
    if kind == "gated_mlp":
        return _tiles((act["silu"](x @ values["w1"]) * (x @ values["w3"])) @ values["w2"])
    hidden = act["gelu"](x @ values["w1"] + pad_bias(values["b1"]))
    return _tiles(_stored(hidden.bfloat16(), "bfp8_b") @ values["w2"] + pad_bias(values["b2"]))


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return _values(ttnn.linear(state["x"], state["w"], bias=state["bias"], activation=state["activation"]))
    if kind == "mlp":
        hidden = tt_lib.tensor.falcon_dense_h_to_4h_matmul(state["x"], state["w1"], fused_activation=tt_lib.tensor.FusibleActivation.GELU)
        return _values(tt_lib.tensor.falcon_dense_4h_to_h_matmul(hidden, state["w2"]))
    if kind == "gated_mlp":
        gate = ttnn.linear(state["x"], state["w1"], activation="silu")
        up = ttnn.linear(state["x"], state["w3"])
        return _values(ttnn.linear(ttnn.mul(gate, up), state["w2"]))
    if kind == "ffn":
        hidden = ttnn.linear(state["x"], state["w1"], bias=state["b1"], activation="gelu", dtype=ttnn.bfloat8_b)
        return _values(ttnn.linear(hidden, state["w2"], bias=state["b2"], dtype=ttnn.bfloat16))
    if kind == "attention":
        return _values(ttnn.matmul(state["q"], state["k_t"])), _values(ttnn.matmul(state["p"], state["v"]))
    if kind == "bmm":
        return _values(ttnn.matmul(state["x"], state["w"]))
    if kind == "from_torch":
        return _values(ttnn.from_torch(state["host"], dtype=state["dtype"], layout=ttnn.TILE_LAYOUT, device=state["device"]))
    return ttnn.to_torch(state["x"])


def _values(tensor):
    """The tensor's own device buffer (tiles), as the next op would read it."""
    return tensor._buf
