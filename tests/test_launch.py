"""Which calls take the eager shortcut around the dispatcher: a small registered op on the CPU in place of the HIP ones."""

from __future__ import annotations

import ctypes

import pytest
import torch

from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from skyrl_amd import _launch
from skyrl_amd._launch import call, raw_stream, registered_op


@registered_op("skyrl_amd_tests::double_it", mutates_args=())
def double_it(x: torch.Tensor) -> torch.Tensor:
    return 2.0 * x.detach()


@double_it.register_fake
def _(x):
    return torch.empty_like(x)


class _Doubled(torch.autograd.Function):
    """As the adapters do it: the op in the forward, where autograd records nothing, and in the backward."""

    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        return call(double_it, x)

    @staticmethod
    def backward(ctx, g):
        (x,) = ctx.saved_tensors
        return call(double_it, g * x)


@pytest.fixture
def route(monkeypatch):
    """The op's shortcut, counted: calls of ``route`` are eager ones."""
    taken = []
    eager = double_it.eager
    monkeypatch.setattr(double_it, "eager", lambda *a: (taken.append(1), eager(*a))[1])
    return taken


def test_plain_calls_take_the_shortcut(route):
    x = torch.ones(3, requires_grad=True)
    assert torch.equal(call(double_it, x.detach()), torch.full((3,), 2.0)) and len(route) == 1
    with torch.no_grad():
        call(double_it, x)
    assert len(route) == 2
    (g,) = torch.autograd.grad(_Doubled.apply(x).sum(), x)  # forward and backward of an ordinary training step
    assert len(route) == 4 and torch.equal(g, torch.full((3,), 2.0))


def test_a_gradient_without_a_formula_raises():
    x = torch.ones(3, requires_grad=True)
    with pytest.raises(RuntimeError, match="no autograd formula"):
        call(double_it, x).sum().backward()
    (g,) = torch.autograd.grad(_Doubled.apply(x).sum(), x, create_graph=True)
    with pytest.raises(RuntimeError, match="no autograd formula"):  # the second derivative is not silently zero
        (x.sum() + g.square().sum()).backward()


@registered_op("skyrl_amd_tests::memory_of", mutates_args=())
def memory_of(x: torch.Tensor) -> torch.Tensor:
    """What a kernel that is given ``x.data_ptr()`` reads."""
    x = x.contiguous()  # the dispatcher expands a zero tensor from one element
    if x.data_ptr() == 0:
        raise RuntimeError("a kernel would read from address 0")
    return torch.frombuffer((ctypes.c_float * x.numel()).from_address(x.data_ptr()), dtype=torch.float32).clone()


def test_tensors_whose_memory_is_not_their_value():
    assert torch.equal(call(memory_of, torch._neg_view(torch.full((3,), 2.0))), torch.full((3,), -2.0))
    assert torch.equal(call(memory_of, torch._efficientzerotensor(3)), torch.zeros(3))


class _WatchDispatch(TorchDispatchMode):
    seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


class _WatchFunctions(TorchFunctionMode):
    seen = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


def test_whoever_follows_the_call_sees_the_op():
    """Tracing, profiling, modes and functorch transforms find the registered op by its name; none of them meets the bare function."""
    x = torch.ones(3)
    double = lambda t: call(double_it, t)  # noqa: E731
    assert "skyrl_amd_tests::double_it" in str(torch.jit.trace(double, x, check_trace=False).inlined_graph)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        double(x)
    assert any("double_it" in e.key for e in prof.key_averages())
    for mode in (_WatchDispatch, _WatchFunctions):
        with mode():
            double(x)
        assert any("double_it" in name for name in mode.seen)
    assert torch.equal(torch.func.vmap(double)(x.reshape(3, 1)), torch.full((3, 1), 2.0))  # by the op's batching fallback


def test_a_torch_without_the_private_counters_takes_the_op(monkeypatch, route):
    monkeypatch.setattr(_launch, "_FOLLOWERS", None)
    assert torch.equal(call(double_it, torch.ones(3)), torch.full((3,), 2.0)) and not route
    monkeypatch.delattr(torch._C, "_is_tracing")
    assert _launch._followers() is None


def test_raw_stream_without_the_private_accessor(monkeypatch):
    class Stream:
        cuda_stream = 77

    monkeypatch.setattr(_launch, "_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev: Stream())
    assert raw_stream(torch.device("cuda", 0)) == 77
