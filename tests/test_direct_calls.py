"""The short way of the package's operators past the dispatcher: taken by plain eager calls only, and equal to the
operator in everything a caller can see."""

import contextlib
import os
import subprocess
import sys

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from flash_model_architectures_amd import ops
from flash_model_architectures_amd.custom_op import _eager, apply_function, direct_xma_op
from flash_model_architectures_amd.functional.routing import _TopkSoftmax


@contextlib.contextmanager
def _dual_level():
    with torch.autograd.forward_ad.dual_level():
        yield


@pytest.mark.parametrize(
    "mode",
    [TorchDispatchMode, TorchFunctionMode, torch.profiler.profile, _dual_level, lambda: torch.device("cpu")],
    ids=["dispatch_mode", "function_mode", "profiler", "forward_mode", "device_context"],
)
def test_observed_calls_are_not_direct(mode):
    assert _eager()
    with mode():
        assert not _eager()
    assert _eager()


@contextlib.contextmanager
def _execution_trace(path):
    observer = torch.profiler.ExecutionTraceObserver().register_callback(str(path))
    observer.start()
    try:
        yield
    finally:
        observer.stop()
        observer.unregister_callback()


def test_execution_trace_holds_every_call(tmp_path):
    """An execution trace observes calls through a callback of its own, without a profiler being enabled."""

    path = tmp_path / "trace.json"
    with _execution_trace(path):
        assert not torch._C._autograd._profiler_enabled() and not _eager()
        apply_function(_Double, torch.ones(3))
        with pytest.raises(RuntimeError, match="ROCm device"):  # the operator is reached, and refuses the host tensor
            ops.swiglu_forward_rocm(*(torch.ones(1, 8) for _ in range(3)))
    trace = path.read_text()
    assert "_Double" in trace and "xma::swiglu_forward_rocm" in trace
    assert _eager()


@pytest.mark.parametrize("name", ["_len_torch_dispatch_stack", "_dispatch_has_kernel_for_any_dispatch_key"])
def test_unknown_predicate_makes_no_call_direct(name):
    """A torch without one of the names that the short way asks: every call takes the long way."""

    program = (
        f"import torch; del torch._C.{name}\n"
        "from flash_model_architectures_amd import ops\n"
        "from flash_model_architectures_amd.custom_op import _eager\n"
        "assert not _eager()\n"
        "try: ops.swiglu_forward_rocm(*(torch.ones(1, 8) for _ in range(3)))\n"
        "except RuntimeError as error: assert 'ROCm device' in str(error)\n"
        "else: raise SystemExit('not refused')\n"
    )
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    done = subprocess.run([sys.executable, "-c", program], cwd=root, capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr


def test_transformed_calls_are_not_direct():
    seen = []

    def observe(x):
        seen.append(_eager())
        return x * 2

    torch.vmap(observe)(torch.ones(2, 3))
    torch.func.grad(lambda x: observe(x).sum())(torch.ones(3))
    torch.func.functionalize(observe)(torch.ones(3))
    make_fx(observe)(torch.ones(3))
    torch.jit.trace(observe, torch.ones(3), check_trace=False)
    assert seen == [False] * len(seen) and len(seen) >= 5


class _Double(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        return x * 2

    @staticmethod
    def backward(ctx, grad):
        return grad * 2


def test_apply_function_records_a_graph_when_one_is_needed():
    x = torch.ones(3, requires_grad=True)
    apply_function(_Double, x).sum().backward()
    assert torch.equal(x.grad, torch.full((3,), 2.0))
    with torch.no_grad():
        assert not apply_function(_Double, x).requires_grad
    assert not apply_function(_Double, x.detach()).requires_grad
    with pytest.raises(RuntimeError, match="setup_context"):  # what autograd says of such a function under a transform
        torch.func.grad(lambda t: apply_function(_Double, t).sum())(x.detach())


class _LongWay(Exception):
    pass


def _refuse(*args, **kwargs):
    raise _LongWay


def test_apply_function_takes_the_short_way(monkeypatch):
    x = torch.ones(3, requires_grad=True)
    monkeypatch.setattr(_Double, "apply", _refuse)
    assert torch.equal(apply_function(_Double, x.detach()), torch.full((3,), 2.0))
    with torch.no_grad():
        assert torch.equal(apply_function(_Double, x), torch.full((3,), 2.0))
    with pytest.raises(_LongWay):
        apply_function(_Double, x)


def _swiglu_arguments(kind: str):
    g = torch.randn(5, 24, device="cuda", dtype=torch.float32, generator=torch.Generator("cuda").manual_seed(1))
    u, y = g.flip(0), torch.zeros_like(g)
    if kind == "negated":  # a lazily negated view: its memory holds the opposite sign
        g = torch.complex(u, -g).conj().imag
        g = g if g.stride(-1) == 1 else torch._neg_view(g.neg())
        assert g.is_neg()
    if kind == "strided":
        wide = torch.zeros(5, 48, device="cuda")
        wide[:, :24] = g
        g = wide[:, :24]
    if kind == "parameter":
        g = torch.nn.Parameter(g, requires_grad=False)
    return g, u, y


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "strided", "parameter", "negated"])
@pytest.mark.parametrize("positional", [False, True])
def test_direct_call_equals_the_operator(kind, positional):
    g, u, y = _swiglu_arguments(kind)
    want = torch.zeros_like(y)
    version = want._version
    ops.swiglu_forward_rocm._custom_op(g, u, want)
    bump = want._version - version
    version = y._version
    assert (ops.swiglu_forward_rocm(g, u, y) if positional else ops.swiglu_forward_rocm(y=y, g=g, u=u)) is None
    assert torch.equal(y, want) and y._version - version == bump == 1


@pytest.mark.gpu
def test_operator_takes_the_short_way(monkeypatch):
    """Which calls reach the operator and which do not."""

    arguments = {kind: _swiglu_arguments(kind) for kind in ("plain", "strided", "parameter", "negated")}
    with torch.inference_mode():
        created_in_inference = tuple(t.clone() for t in arguments["plain"])
    monkeypatch.setattr(type(ops.swiglu_forward_rocm._custom_op), "__call__", _refuse)
    for kind in ("plain", "strided", "parameter"):
        ops.swiglu_forward_rocm(*arguments[kind])
        ops.swiglu_forward_rocm(**dict(zip("guy", arguments[kind])))
    g, u, y = arguments["plain"]
    with torch.inference_mode():
        ops.swiglu_forward_rocm(*arguments["plain"])
        ops.swiglu_forward_rocm(*created_in_inference)
    differentiable = g.clone().requires_grad_()
    with torch.no_grad():
        ops.swiglu_forward_rocm(differentiable, u, y)
    for long in (
        lambda: ops.swiglu_forward_rocm(*arguments["negated"]),
        lambda: ops.swiglu_forward_rocm(differentiable, u, y),
        lambda: ops.swiglu_forward_rocm(*created_in_inference),  # outputs of inference mode outside it
        lambda: ops.swiglu_forward_rocm(g, u.cpu(), y),
        lambda: ops.swiglu_forward_rocm(g, u, 1.0),
        lambda: ops.swiglu_forward_rocm(g, u, y, y),
    ):
        with pytest.raises(_LongWay):
            long()


def _register_in_library(key):
    def register(op, kernel):
        library = torch.library.Library("xma", "IMPL")
        library.impl(op.__name__, kernel, key)
        return library._destroy

    return register


def _register_in_definition(device):
    return lambda op, kernel: op._custom_op.register_kernel(device)(kernel)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "name,register",
    [
        ("library_device", _register_in_library("CUDA")),
        ("library_autograd", _register_in_library("AutogradCUDA")),
        ("definition", _register_in_definition(None)),
        ("definition_device", _register_in_definition("cuda")),
    ],
)
def test_registered_kernel_is_called(name, register):
    """A kernel that a program registers for an operator is called, and no longer once its library is gone."""

    def copy(x: "torch.Tensor", y: "torch.Tensor") -> None:
        y.copy_(x)

    copy.__name__ = f"test_copy_{name}"
    op, calls = direct_xma_op(mutates_args={"y"})(copy), []
    x, y = torch.ones(4, device="cuda"), torch.zeros(4, device="cuda")
    undo = register(op, lambda x, y: calls.append(y))
    op(x, y)
    assert len(calls) == 1 and not y.any()
    if name.startswith("library"):
        undo()
        op(x, y)
        assert len(calls) == 1 and torch.equal(x, y)


@pytest.mark.gpu
def test_overwritten_saved_tensor_is_still_noticed():
    g, u, y = _swiglu_arguments("plain")
    w = torch.ones_like(y, requires_grad=True)
    product = w * y  # saves y for the backward
    ops.swiglu_forward_rocm(g=g, u=u, y=y)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        product.sum().backward()


@pytest.mark.gpu
def test_wrong_arguments_are_refused():
    g, u, y = _swiglu_arguments("plain")
    logits, weights = torch.randn(4, 8, device="cuda"), torch.empty(4, 2, device="cuda")
    indices = torch.empty(4, 2, dtype=torch.int64, device="cuda")
    for refused in (
        lambda: ops.swiglu_forward_rocm(g, u),
        lambda: ops.swiglu_forward_rocm(g, u, y, y),
        lambda: ops.swiglu_forward_rocm(g, u, out=y),
        lambda: ops.swiglu_forward_rocm(g, u.cpu(), y),
        lambda: ops.topk_softmax_rocm(logits, weights, indices, 2.0),
        lambda: ops.topk_softmax_rocm(logits, weights, indices, "2"),
    ):
        with pytest.raises((RuntimeError, TypeError, ValueError)):
            refused()


@pytest.mark.gpu
def test_inference_mode_and_profiler():
    g, u, y = _swiglu_arguments("plain")
    ops.swiglu_forward_rocm(g=g, u=u, y=y)
    with torch.inference_mode():
        z = torch.zeros_like(y)
        ops.swiglu_forward_rocm(g=g, u=u, y=z)
        weights, indices = apply_function(_TopkSoftmax, torch.randn(4, 8, device="cuda"), 2, torch.int64)
        assert weights.is_inference() and indices.is_inference()
    assert torch.equal(y, z)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
        ops.swiglu_forward_rocm(g=g, u=u, y=y)
    assert any(event.key == "xma::swiglu_forward_rocm" for event in profile.key_averages())
