"""Which calls take the eager shortcut around the dispatcher: a small registered op on the CPU in place of the HIP ones."""

from __future__ import annotations

import ctypes

import pytest
import torch

from skyrl_amd._launch import call, registered_op


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
