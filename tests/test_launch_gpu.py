"""The eager shortcut around the dispatcher gives what the registered op gives, and steps aside where a dispatch mode or a tensor
subclass has to see the op."""

from __future__ import annotations

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from skyrl_amd import ops
from skyrl_amd._launch import call

pytestmark = pytest.mark.gpu


def test_call_is_the_op_and_lets_modes_and_fake_tensors_see_it(cuda_device):
    T, H, V = 40, 64, 300
    gen = torch.Generator().manual_seed(0)
    args = (torch.randn(T, H, generator=gen).bfloat16().to(cuda_device), torch.randn(V, H, generator=gen).bfloat16().to(cuda_device),
            torch.randint(0, V, (T,), generator=gen).to(cuda_device), 1.0, True)
    for got, want in zip(call(ops.lmhead_fwd, *args), ops.lmhead_fwd(*args)):
        assert torch.equal(got, want)

    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, a=(), kw=None):
            seen.append(str(func))
            return func(*a, **(kw or {}))

    with Watch():
        call(ops.lmhead_fwd, *args)
    assert any("skyrl_amd.lmhead_fwd" in s for s in seen)
    with FakeTensorMode() as mode:
        fake = call(ops.lmhead_fwd, *(mode.from_tensor(a) if isinstance(a, torch.Tensor) else a for a in args))
    assert [tuple(t.shape) for t in fake] == [(T,)] * 4 and all(type(t) is not torch.Tensor for t in fake)
