"""The workloads this package is timed on: what a program that uses the Mixture-of-Experts path has it do.

Five families, each over the range its users have:

* `moe`, forward (serving): from one decoded token to a long prompt;
* `moe`, training: forward and backward, from micro-batches of a few hundred tokens to full batches;
* `swiglu`: the gated activation on its own, forward and backward, as a dense MLP calls it;
* `packing`: padding taken out of a batch and put back, forward and backward;
* `routing`: expert histogram and stable permutation of a stream of expert ids.

Expert shapes are the three of the benchmark (Mixtral-shaped, fine-grained, skewed), those of the layer's test
matrix, and generic ones.
"""

from __future__ import annotations

import math

import torch
import torch.nn as nn

import flash_model_architectures_amd as xma


DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# (hidden, intermediate, experts, experts per token)
MIXTRAL_SHAPED = (4096, 14336, 8, 2)
FINE_GRAINED = (2048, 1024, 64, 6)
MANY_EXPERTS = (2048, 768, 128, 8)
TEST_MATRIX = [(2048, 8192, 2, 2), (2048, 8192, 8, 4), (512, 1024, 4, 2), (512, 1024, 6, 4), (576, 256, 128, 8)]

LARGEST_FLOPS = 18 * 8192 * 2 * 4096 * 14336  # the Mixtral-shaped training step
LARGEST_PARAMETERS = 3 * 8 * 4096 * 14336 * 2  # bytes of its expert weights
FP32_COST = 16  # ratio of the dense bf16 and fp32 matrix rates
UNALIGNED_COST = 8  # sizes that are not multiples of the vector width leave the vector loads


def _moe(name, train, tokens, shape, dtype="bf16", activation="swiglu_packed", bias=False, skewed=False):
    hidden, intermediate, experts, top_k = shape
    case = {
        "family": "moe",
        "train": train,
        "tokens": tokens,
        "hidden": hidden,
        "intermediate": intermediate,
        "experts": experts,
        "top_k": top_k,
        "dtype": dtype,
        "activation": activation,
        "bias": bias,
        "skewed": skewed,
    }
    return case if name is None else {"name": name, **case}


def listed() -> list[dict]:
    return [
        # one sequence being decoded on a fine-grained layer: the smallest call there is, six experts' weights and latency
        _moe("decode_one_token", False, 1, FINE_GRAINED),
        # a serving batch being decoded on the Mixtral-shaped layer: every expert is hit by a few tokens
        _moe("decode_batch", False, 32, MIXTRAL_SHAPED),
        # a prompt of no particular length through a layer whose router favours a few experts
        _moe("prefill_skewed", False, 1531, MANY_EXPERTS, skewed=True),
        # evaluation of a small full-precision layer
        _moe("forward_small_fp32", False, 1024, (256, 512, 8, 2), dtype="fp32"),
        # a small training step with a plain activation and expert biases, token count and rows per expert ragged
        _moe("train_small_fp16", True, 3001, (512, 1024, 6, 4), dtype="fp16", activation="gelu_tanh", bias=True),
        # full training steps of the three benchmark layers
        _moe("train_mixtral_shaped", True, 8192, MIXTRAL_SHAPED),
        _moe("train_fine_grained", True, 16384, FINE_GRAINED),
        _moe("train_skewed", True, 16384, MANY_EXPERTS, skewed=True),
        # full-precision training of a layer of the test matrix
        _moe("train_fp32", True, 2048, (2048, 8192, 8, 4), dtype="fp32"),
        # the activation of a dense MLP at the Mixtral width, forward and backward
        {"name": "swiglu_step", "family": "swiglu", "rows": 16384, "cols": 14336, "dtype": "bf16"},
        # a padded batch to packed tokens and back, forward and backward, three quarters full
        {
            "name": "packing_step",
            "family": "packing",
            "batch": 16,
            "length": 4096,
            "hidden": 4096,
            "dtype": "bf16",
            "padding_side": "left",
        },
        # counting and grouping a large batch's expert choices
        {"name": "routing", "family": "routing", "ids": 1 << 20, "experts": 256, "index": "int32"},
    ]


def _log_int(rng, low: int, high: int) -> int:
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _draw_shape(rng) -> tuple[int, int, int, int]:
    which = rng.random()
    if which < 0.45:
        return rng.choice([MIXTRAL_SHAPED, FINE_GRAINED, MANY_EXPERTS])
    if which < 0.7:
        return rng.choice(TEST_MATRIX)
    hidden = 8 * _log_int(rng, 32, 512)
    intermediate = 8 * _log_int(rng, 32, 1024)
    if rng.random() < 0.1:  # nothing a multiple of the vector width
        hidden, intermediate = hidden // 8 + 1, intermediate // 8 + 3
    experts = rng.choice([4, 6, 8, 16, 32, 64, 128])
    return hidden, intermediate, experts, rng.choice([k for k in (1, 2, 4, 6, 8) if k <= experts])


def _draw_moe(rng, train: bool) -> dict:
    while True:
        tokens = _log_int(rng, 64 if train else 1, 16384)
        case = _moe(
            None,
            train,
            tokens,
            _draw_shape(rng),
            dtype=rng.choices(["bf16", "fp16", "fp32"], [6, 2, 2])[0],
            activation=rng.choices(["swiglu_packed", "glu", "gelu_tanh", "silu"], [6, 1, 2, 1])[0],
            bias=rng.random() < 0.2,
            skewed=rng.random() < 0.25,
        )
        cost = work(case)["flops"]
        cost *= FP32_COST if case["dtype"] == "fp32" else 1
        cost *= UNALIGNED_COST if case["hidden"] % 8 or case["intermediate"] % 8 else 1
        parameters = 3 * case["experts"] * case["hidden"] * case["intermediate"] * DTYPES[case["dtype"]].itemsize
        if cost <= LARGEST_FLOPS and parameters <= LARGEST_PARAMETERS:
            return case


def draw(rng) -> dict:
    family = rng.choices(["serve", "train", "swiglu", "packing", "routing"], [4, 4, 1, 1, 1])[0]
    if family == "serve":
        return _draw_moe(rng, False)
    if family == "train":
        return _draw_moe(rng, True)
    if family == "swiglu":
        cols = rng.choice([1024, 4096, 14336, 8 * _log_int(rng, 16, 2048), _log_int(rng, 100, 5000)])
        return {
            "family": "swiglu",
            "rows": _log_int(rng, 1, max(1, 16384 * 14336 // cols)),
            "cols": cols,
            "dtype": rng.choice(["bf16", "fp16", "fp32"]),
        }
    if family == "packing":
        batch, length = rng.randint(1, 32), _log_int(rng, 16, 4096)
        hidden = rng.choice([512, 4096, 8 * _log_int(rng, 8, 512), _log_int(rng, 33, 1000)])
        while batch * length * hidden > 16 * 4096 * 4096:
            batch = max(1, batch // 2)
            length = length if batch > 1 else length // 2
        return {
            "family": "packing",
            "batch": batch,
            "length": length,
            "hidden": hidden,
            "dtype": rng.choice(["bf16", "fp16", "fp32"]) if batch * length * hidden <= 8 * 4096 * 4096 else "bf16",
            "padding_side": rng.choice(["left", "right"]),
        }
    return {
        "family": "routing",
        "ids": _log_int(rng, 8, 1 << 22),
        "experts": rng.choice([2, 8, 60, 64, 128, 256, 384, 1000]),
        "index": rng.choice(["int32", "int64"]),
    }


# ---- inputs -------------------------------------------------------------------------------------------------------


def _activation(name: str):
    """(callable handed to the layer, whether it halves its input)"""

    if name == "swiglu_packed":
        return xma.swiglu_packed, True
    if name == "glu":
        return nn.GLU(), True
    if name == "gelu_tanh":
        return nn.GELU(approximate="tanh"), False
    return nn.SiLU(), False


def _prepare_moe(case: dict, generator: torch.Generator, seed: int) -> dict:
    dtype = DTYPES[case["dtype"]]
    activation, is_glu = _activation(case["activation"])
    torch.manual_seed(seed)  # parameters are drawn by the module itself
    with torch.device("cuda"):
        layer = xma.MoE(
            case["experts"], case["top_k"], case["hidden"], case["intermediate"], activation, is_glu, case["bias"], 0.02
        )
    x = torch.randn(case["tokens"], case["hidden"], device="cuda", generator=generator)
    with torch.no_grad():
        if case["bias"]:
            for projection in (layer.c_fc, layer.c_proj):
                projection.bias.normal_(0, 0.02)
        if case["skewed"]:
            # one feature is the same for every token, and the router's weight on it falls like Zipf's law (s = 1.2)
            # over the experts: a few experts take most of the rows and many take none
            x[:, 0] = 1.0
            ranks = torch.arange(1, case["experts"] + 1, device="cuda", dtype=torch.float32)
            layer.gate.weight[:, 0] = -1.2 * ranks.log()
    layer = layer.to(dtype)
    state = {"layer": layer, "x": x.to(dtype)}
    if case["train"]:
        state["x"].requires_grad_()
        state["dy"] = torch.randn(x.shape, device="cuda", generator=generator).to(dtype)
    else:
        layer.requires_grad_(False).eval()
    return state


def _lengths(case: dict) -> list[int]:
    """Sequence lengths spread evenly from half full to full: three quarters of the padded length on average."""

    batch, length = case["batch"], case["length"]
    return [length - (length // 2) * b // max(1, batch - 1) for b in range(batch)]


def prepare(case: dict, seed: int) -> dict:
    generator = torch.Generator(device="cuda").manual_seed(seed)
    family = case["family"]
    if family == "moe":
        state = _prepare_moe(case, generator, seed)
    elif family == "swiglu":
        dtype = DTYPES[case["dtype"]]
        x = torch.randn(case["rows"], 2 * case["cols"], device="cuda", generator=generator).to(dtype)
        dy = torch.randn(case["rows"], case["cols"], device="cuda", generator=generator).to(dtype)
        state = {"x": x.requires_grad_(), "dy": dy}
    elif family == "packing":
        dtype = DTYPES[case["dtype"]]
        lengths = torch.tensor(_lengths(case), device="cuda")
        order = torch.randperm(case["batch"], device="cuda", generator=generator)  # sequences come in any order
        cu_seqlens = torch.zeros(case["batch"] + 1, dtype=torch.int32, device="cuda")
        cu_seqlens[1:] = lengths[order].cumsum(0)
        shape = (case["batch"], case["length"], case["hidden"])
        x = torch.randn(shape, device="cuda", generator=generator).to(dtype)
        dy = torch.randn(shape, device="cuda", generator=generator).to(dtype)
        # a data loader knows the token count on the host
        state = {"x": x.requires_grad_(), "dy": dy, "cu_seqlens": cu_seqlens, "total": sum(_lengths(case))}
    else:
        # choices of a router with a mild preference: the density falls linearly over the expert index
        u = torch.rand(case["ids"], device="cuda", generator=generator)
        ids = ((1.0 - u.sqrt()) * case["experts"]).to(torch.int64).clamp_(0, case["experts"] - 1)
        state = {"ids": ids.to(torch.int32 if case["index"] == "int32" else torch.int64)}
    state["case"] = case
    return state


# ---- one pass -----------------------------------------------------------------------------------------------------


def _run_moe(state: dict) -> dict:
    layer, x = state["layer"], state["x"]
    if not state["case"]["train"]:
        with torch.no_grad():
            y, logits = layer(x)
        return {"y": y, "router_logits": logits}
    layer.zero_grad(set_to_none=True)
    x.grad = None
    y, logits = layer(x)
    y.backward(state["dy"])
    gradients = {f"d {name}": parameter.grad for name, parameter in layer.named_parameters()}
    return {"y": y.detach(), "router_logits": logits.detach(), "d x": x.grad, **gradients}


def run(state: dict) -> dict:
    case = state["case"]
    family = case["family"]
    if family == "moe":
        return _run_moe(state)
    if family == "swiglu":
        x = state["x"]
        x.grad = None
        y = xma.swiglu_packed(x)
        y.backward(state["dy"])
        return {"y": y.detach(), "d x": x.grad}
    if family == "packing":
        x = state["x"]
        x.grad = None
        side = case["padding_side"]
        (packed,) = xma.pack_sequence([x], state["cu_seqlens"], state["total"], side)
        (padded,) = xma.unpack_sequence([packed], state["cu_seqlens"], case["batch"], case["length"], side)
        padded.backward(state["dy"])
        return {"packed": packed.detach(), "padded": padded.detach(), "d x": x.grad}
    counts = xma.continuous_count(state["ids"], case["experts"])
    routing = xma.route_tokens(state["ids"], case["experts"])
    return {
        "counts": counts,
        "expert_frequency": routing.expert_frequency,
        "expert_offsets": routing.expert_offsets,
        "sorted_expert_idxs": routing.sorted_expert_idxs,
        "sorted_scattered_idxs": routing.sorted_scattered_idxs,
    }


# ---- what a pass cannot do without ----------------------------------------------------------------------------------


def _experts_hit(case: dict) -> float:
    """Experts that receive a token, on average."""

    T, E, k = case["tokens"], case["experts"], case["top_k"]
    if not case["skewed"]:
        return E * (1.0 - (1.0 - k / E) ** T)
    # the logits of a freshly initialised router have a variance of 1/3; see _prepare_moe for the skew
    logits = torch.randn(T, E, generator=torch.Generator().manual_seed(0)) / math.sqrt(3.0)
    logits -= 1.2 * torch.arange(1, E + 1, dtype=torch.float32).log()
    return float(logits.topk(k).indices.unique().numel())


def _work_moe(case: dict) -> dict:
    T, H, I, E, k = (case[n] for n in ("tokens", "hidden", "intermediate", "experts", "top_k"))
    size = DTYPES[case["dtype"]].itemsize
    _, is_glu = _activation(case["activation"])
    up = 2 * I if is_glu else I
    rows = T * k
    expert = H * (up + I) + ((up + H) if case["bias"] else 0)  # parameters of one expert
    hit = _experts_hit(case)
    forward_flops = 2 * rows * H * (up + I) + 2 * T * H * E
    forward_bytes = size * (2 * T * H + T * E + E * H + hit * expert)
    if not case["train"]:
        return {"bytes": forward_bytes, "flops": forward_flops}
    # gradients: dy read, dx written, every parameter's gradient written (those of experts without tokens too)
    return {"bytes": forward_bytes + size * (2 * T * H + E * H + E * expert), "flops": 3 * forward_flops}


def work(case: dict) -> dict:
    family = case["family"]
    if family == "moe":
        return _work_moe(case)
    if family == "swiglu":
        n = case["rows"] * case["cols"]
        # x (two halves), dy read; y, dx (two halves) written; sigmoid, three products and their gradients
        return {"bytes": 6 * n * DTYPES[case["dtype"]].itemsize, "flops": 20 * n}
    if family == "packing":
        row = case["hidden"] * DTYPES[case["dtype"]].itemsize
        padded, packed = case["batch"] * case["length"] * row, sum(_lengths(case)) * row
        # x read where it is not padding, packed written, padded written; dy read, dx written
        return {"bytes": 2 * packed + padded + packed + padded, "flops": 0}
    index = 4 if case["index"] == "int32" else 8
    # ids read, two int32 tables written
    return {"bytes": case["ids"] * (index + 8) + 12 * case["experts"], "flops": 0}


def tolerance(case: dict):
    """About four times the largest difference of any output from the same path in 64-bit floating point on the same
    expert choices: measured 5.1e-3 / 5.7e-4 / 2.5e-6 for the layer in bf16 / fp16 / fp32 (the input gradient is the
    worst everywhere, sizes and activations matter little) and 1.7e-3 / 2.1e-4 / 5.2e-8 for SwiGLU alone.  Moves and
    integers are exact."""

    if case["family"] in ("packing", "routing"):
        return "exact"
    if case["family"] == "swiglu":
        return {"rel": {"bf16": 7e-3, "fp16": 8.5e-4, "fp32": 2.5e-7}[case["dtype"]]}
    return {"rel": {"bf16": 2e-2, "fp16": 2.3e-3, "fp32": 1e-5}[case["dtype"]]}
