"""The experts of a layer from one native call: the same results, bit for bit, as the operators one by one, and the operators
whenever a call is not a plain one."""

import threading

import pytest
import torch
import torch.nn as nn
from torch.utils._python_dispatch import TorchDispatchMode
from torch.utils.checkpoint import checkpoint

import flash_model_architectures_amd as xma
from flash_model_architectures_amd import _native, ops
from flash_model_architectures_amd.functional import routing as routing_module
from flash_model_architectures_amd.layers import moe
from oracle import torch_oracle as to

from .helpers import TOL, assert_close


ACTIVATIONS = {
    "swiglu": (xma.swiglu_packed, True),
    "glu": (nn.GLU(), True),
    "gelu_tanh": (nn.GELU(approximate="tanh"), False),
}


def _layer(dtype, activation="swiglu", bias=False, experts=6, k=4, hidden=136, intermediate=72):
    torch.manual_seed(0)
    function, is_glu = ACTIVATIONS[activation]
    layer = xma.MoE(experts, k, hidden, intermediate, function, is_glu, bias, 0.05)
    if bias:
        with torch.no_grad():
            layer.c_fc.bias.normal_()
            layer.c_proj.bias.normal_()
    return layer.to("cuda").to(dtype)


def _layer_on_cpu():
    return xma.MoE(4, 2, 16, 8, xma.swiglu_packed, True, False, 0.05)


def _train(layer, x, dy):
    layer.zero_grad(set_to_none=True)
    x = x.detach().requires_grad_()
    y, logits = layer(x)
    y.backward(dy)
    return [y.detach(), logits.detach(), x.grad, *(p.grad for p in layer.parameters())]


class _Calls:
    """Native entry points called, in order."""

    def __init__(self, monkeypatch, one_by_one=False):
        self.names = []
        real = _native.load()
        calls = self

        class Library:
            def __getattr__(self, name):
                if name in ("xma_moe_forward", "xma_moe_backward"):
                    calls.names.append(name)
                return getattr(real, name)

        monkeypatch.setattr(_native, "_lib", Library())
        if one_by_one:
            monkeypatch.setattr(_native, "_timeline", _native.Timeline())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("activation", list(ACTIVATIONS))
@pytest.mark.parametrize("tokens,sizes", [(1, {}), (67, {}), (300, dict(k=1)), (40, dict(hidden=33, intermediate=21))])
def test_same_results(tokens, sizes, activation, bias, dtype, monkeypatch):
    layer = _layer(dtype, activation, bias, **sizes)
    x = torch.randn(tokens, layer.hidden_size, device="cuda", dtype=dtype)
    dy = torch.randn_like(x)
    results = {}
    for one_by_one in (False, True):
        with monkeypatch.context() as patch:
            calls = _Calls(patch, one_by_one)
            with torch.no_grad():
                forward = layer(x)
            results[one_by_one] = [*forward, *_train(layer, x, dy)]
            assert calls.names == ([] if one_by_one else ["xma_moe_forward", "xma_moe_forward", "xma_moe_backward"])
    for a, b in zip(results[False], results[True]):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_calls_that_are_not_plain(monkeypatch):
    layer = _layer(torch.bfloat16)
    x = torch.randn(50, layer.hidden_size, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        want = layer(x)[0]

    class Seen(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_dispatch__(self, function, types, args=(), kwargs=None):
            self.names.append(str(function))
            return function(*args, **(kwargs or {}))

    calls = _Calls(monkeypatch)
    with torch.no_grad(), Seen() as seen:
        assert torch.equal(layer(x)[0], want)
    assert any("topk_softmax" in name for name in seen.names) and any("up_projection" in name for name in seen.names)
    assert calls.names == []

    # a step that a program has replaced is called
    replaced = []

    def routing(hidden_states, *, kernel_backend=None):
        replaced.append(hidden_states.shape)
        return xma.MoE._compute_routing_weights(layer, hidden_states, kernel_backend=kernel_backend)

    layer._compute_routing_weights = routing
    with torch.no_grad():
        assert torch.equal(layer(x)[0], want)
    assert replaced == [x.shape]
    del layer._compute_routing_weights

    # weights that are views of other storage
    storage = layer.c_fc.weight.detach().transpose(1, 2).contiguous()
    layer.c_fc.weight = nn.Parameter(storage.transpose(1, 2))
    calls.names.clear()
    with torch.no_grad():
        with pytest.raises(AssertionError):
            layer(x)  # as the operator has always judged such weights
    assert calls.names == []


@pytest.mark.gpu
def test_inference_mode_and_streams():
    layer = _layer(torch.bfloat16)
    x = torch.randn(50, layer.hidden_size, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        want = layer(x)[0]
    with torch.inference_mode():
        assert torch.equal(layer(x.clone())[0], want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), torch.cuda.stream(side):
        on_side = [layer(x)[0] for _ in range(3)]
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(y, want) for y in on_side)


@pytest.mark.gpu
def test_bad_arguments_are_refused():
    args = _native.MOE_ARGS.pack(8, *[0] * (5 + 3 + 17 + 1 + 10))
    assert _native.load().xma_moe_forward(args, 0) != 0 and "bad args" in _native.last_error()
    args = _native.MOE_ARGS.pack(_native.MOE_ARGS.size, 0, ops.nat.EPI_SWIGLU, 4, 2, 0, 1, 8, 8, *[0] * (17 + 1 + 10))
    assert _native.load().xma_moe_backward(args, 0) != 0 and "null pointer" in _native.last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens", [4003, 4800])
def test_gathered_weight_gradient_of_large_tiles(tokens, dtype, monkeypatch):
    """The up-projection's weight gradient reads the tokens where they are, in 256 x 256 tiles too (the rest of this file has
    128 x 128 ones), with part-full last tiles and reductions that end anywhere."""

    layer = _layer(dtype, experts=16, k=2, hidden=1032, intermediate=1032)
    x = torch.randn(tokens, 1032, device="cuda", dtype=dtype)
    dy = torch.randn_like(x)
    want = None
    for one_by_one in (True, False):
        with monkeypatch.context() as patch:
            calls = _Calls(patch, one_by_one)
            got = _train(layer, x, dy)
            assert len(calls.names) == (0 if one_by_one else 2)
        if want is not None:
            for a, b in zip(got, want):
                assert torch.equal(a, b)
        want = got


STEPS = ["_compute_routing_weights", "_compute_experts"]
# names by which the layer's module calls what a native call stands for, and whether the forward pass calls them
NAMES = {
    **dict.fromkeys(["_FusedExperts", "topk_softmax", "route_tokens", "up_projection_fused", "scatter2scatter", "combine_topk"], True),
    **dict.fromkeys(
        ["invert_index", "spread_rows_gate_grad", "spread_rows", "expert_colsum", "group_bwd_W", "down_projection_dgrad_fused"], False
    ),
}
BOTH = ("scatter2scatter", "combine_topk")  # called in both directions


def test_replaced_steps_are_not_own(monkeypatch):
    layer = _layer_on_cpu()
    assert layer._steps_are_own()
    for name in STEPS:
        with monkeypatch.context() as patch:
            patch.setattr(xma.MoE, name, lambda *args, **kwargs: None)
            assert not layer._steps_are_own()
    for name, forward in NAMES.items():
        with monkeypatch.context() as patch:
            patch.setattr(moe, name, object())
            assert layer._steps_are_own() is not forward
            assert (moe._backward_operators() == moe._OWN_BACKWARD_OPERATORS) is (forward and name not in BOTH)
    for name in ("topk_softmax_rocm", "route_build_rocm"):
        with monkeypatch.context() as patch:
            patch.setattr(routing_module, name, object())
            assert not layer._steps_are_own()
    assert layer._steps_are_own()


@pytest.mark.gpu
@pytest.mark.parametrize("step", STEPS)
def test_steps_replaced_on_the_class(step, monkeypatch):
    layer = _layer(torch.bfloat16)
    x = torch.randn(50, layer.hidden_size, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        want = layer(x)[0]
    own, called = getattr(xma.MoE, step), []

    def replaced(self, *args, **kwargs):
        called.append(step)
        return own(self, *args, **kwargs)

    monkeypatch.setattr(xma.MoE, step, replaced)
    with torch.no_grad():
        assert torch.equal(layer(x)[0], want)
    assert len(called) == 1
    assert torch.equal(layer(x)[0], want)
    assert len(called) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("name", [name for name in NAMES if name != "_FusedExperts"])
def test_replaced_names_are_called(name, monkeypatch):
    layer = _layer(torch.bfloat16, bias=True)
    x = torch.randn(50, layer.hidden_size, device="cuda", dtype=torch.bfloat16)
    dy = torch.randn_like(x)
    with torch.no_grad():
        want = layer(x)[0]
    gradients = _train(layer, x, dy)
    own, called = getattr(moe, name), []

    def replaced(*args, **kwargs):
        called.append(name)
        return own(*args, **kwargs)

    monkeypatch.setattr(moe, name, replaced)
    if NAMES[name]:
        with torch.no_grad():
            assert torch.equal(layer(x)[0], want)
        assert called
        called.clear()
    for a, b in zip(_train(layer, x, dy), gradients):
        assert torch.equal(a, b)
    assert called


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_saved_tensor_hooks_and_checkpoints(dtype, monkeypatch):
    """What a call keeps for its backward pass may be replaced by copies, or be made again there."""

    layer = _layer(dtype, bias=True)
    x = torch.randn(77, layer.hidden_size, device="cuda", dtype=dtype)
    dy = torch.randn_like(x)
    want = _train(layer, x, dy)
    packed = []

    def pack(t):
        packed.append(t.shape)
        return t.cpu()

    calls = _Calls(monkeypatch)
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
        got = _train(layer, x, dy)
    assert len(packed) >= 9 and calls.names == ["xma_moe_forward", "xma_moe_backward"]
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    for reentrant in (False, True):
        calls.names.clear()
        layer.zero_grad(set_to_none=True)
        leaf = x.detach().requires_grad_()
        y, _ = checkpoint(layer, leaf, use_reentrant=reentrant)
        y.backward(dy)
        assert calls.names == ["xma_moe_forward", "xma_moe_forward", "xma_moe_backward"]
        for a, b in zip([y.detach(), leaf.grad, *(p.grad for p in layer.parameters())], [want[0], *want[2:]]):
            assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("forward_on_side", [False, True])
def test_directions_on_different_streams(forward_on_side):
    layer = _layer(torch.bfloat16)
    x = torch.randn(900, layer.hidden_size, device="cuda", dtype=torch.bfloat16)
    dy = torch.randn_like(x)
    want = _train(layer, x, dy)
    main, side = torch.cuda.current_stream(), torch.cuda.Stream()
    first, second = (side, main) if forward_on_side else (main, side)
    for _ in range(3):
        layer.zero_grad(set_to_none=True)
        leaf = x.detach().requires_grad_()
        first.wait_stream(main)
        with torch.cuda.stream(first):
            y, _ = layer(leaf)
        second.wait_stream(first)
        with torch.cuda.stream(second):
            y.backward(dy)
        main.wait_stream(side)
        for a, b in zip([y.detach(), leaf.grad, *(p.grad for p in layer.parameters())], [want[0], *want[2:]]):
            assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_two_threads_train_on_one_stream(dtype):
    """One thread's forward pass beside the other's backward one, which runs in a thread of autograd's."""

    layers = [_layer(dtype, experts=6, k=2, hidden=512, intermediate=256), _layer(dtype, experts=200, k=4)]
    work = []
    for layer in layers:
        x = torch.randn(1500, layer.hidden_size, device="cuda", dtype=dtype)
        dy = torch.randn_like(x)
        work.append((layer, x, dy, _train(layer, x, dy)))
    failures = []

    def loop(layer, x, dy, want):
        try:
            for _ in range(20):
                assert all(torch.equal(a, b) for a, b in zip(_train(layer, x, dy), want))
        except BaseException as e:  # noqa: BLE001 (handed to the main thread)
            failures.append(e)

    threads = [threading.Thread(target=loop, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [300_001, 540_001])
def test_many_token_bytes(tokens, monkeypatch):
    """Token rows more than 2^31 bytes behind the first one, whose offsets fill 32 bits, and beyond 2^32, where the rows are
    copied."""

    layer = _layer(torch.bfloat16, experts=8, k=1, hidden=4096, intermediate=64)
    assert (tokens * 4096 * 2 < 2**32) is (tokens == 300_001)
    x = torch.randn(tokens, 4096, device="cuda", dtype=torch.bfloat16)
    dy = torch.randn_like(x)
    want = None
    for one_by_one in (True, False):
        with monkeypatch.context() as patch:
            calls = _Calls(patch, one_by_one)
            got = _train(layer, x, dy)
            assert len(calls.names) == (0 if one_by_one else 2)
        if want is not None:
            for a, b in zip(got, want):
                assert torch.equal(a, b)
        want = got
    # and the last tokens' part in a weight gradient: their experts' gradients change with them
    del want
    x[-1].zero_()
    assert not all(torch.equal(a, b) for a, b in zip(got[3:], _train(layer, x, dy)[3:]))


@pytest.mark.gpu
@pytest.mark.parametrize(
    "tokens,sizes,copied",
    [
        (620, dict(intermediate=256), True),  # 413 rows per expert, 512 columns
        (700, dict(intermediate=252), False),  # 466 rows, 504 columns
        (160, dict(intermediate=1024), True),  # 107 rows, 2048 columns
        (560, dict(k=1, intermediate=256), False),  # 93 rows
    ],
)
def test_token_rows_of_the_fp32_weight_gradient(tokens, sizes, copied, monkeypatch):
    """Long reductions of wide gradients read a copy of the tokens' rows, others look them up: the same sums."""

    sizes = {"intermediate": 256, **sizes}
    layer = _layer(torch.float32, experts=6, hidden=136, **sizes)
    rows, columns = tokens * layer.top_k / 6, 2 * sizes["intermediate"]
    assert copied is (columns >= 512 and rows * columns >= 200000)
    x = torch.randn(tokens, 136, device="cuda")
    dy = torch.randn_like(x)
    want = _train(layer, x, dy)
    calls = _Calls(monkeypatch, one_by_one=True)
    got = _train(layer, x, dy)
    assert calls.names == []
    launched = [tag for tag, *_ in _native._timeline.records]
    assert launched.count("xma_spread_rows") == (1 if copied else 0)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    # against float64
    double = [p.detach().cpu().double().requires_grad_() for p in layer.parameters()]  # gate, up, down
    y, _ = to.moe_forward(x.cpu().double(), *double, layer.top_k)
    y.backward(dy.cpu().double())
    assert_close(got[4].cpu(), double[1].grad.float(), TOL[torch.float32], "dW_up")
