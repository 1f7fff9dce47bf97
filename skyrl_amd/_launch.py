"""Host side of a launch: the registered ops called without the dispatcher where nothing can tell the difference, the current
stream as an integer, and a device guard that costs nothing when the device is already current.

A ``torch.library`` op is what tracing, fake tensors and dispatch modes see; in a plain eager call its dispatcher layers only add
time, 20 to 30 microseconds each, which a scoring pass of 100 microseconds or a chain of small loss kernels does not hide.
"""

from __future__ import annotations

import contextlib

import torch

__all__ = ["registered_op", "plain_eager", "call", "device_guard", "raw_stream"]

_PLAIN = (torch.Tensor, torch.nn.Parameter)
_NO_GUARD = contextlib.nullcontext()


def _followers():
    """torch's private counters of who follows a call, or None where this torch has them under other names."""
    try:
        return (torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack, torch._C._functorch.peek_interpreter_stack,
                torch._C._is_tracing, torch._C._autograd._profiler_enabled, torch.Tensor._is_zerotensor)
    except AttributeError:
        return None


_FOLLOWERS = _followers()
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def registered_op(name: str, mutates_args=()):
    """``torch.library.custom_op`` that keeps the function it registers as ``op.eager``."""
    def register(fn):
        op = torch.library.custom_op(name, mutates_args=mutates_args)(fn)
        op.eager = fn
        return op
    return register


def plain_eager() -> bool:
    """Whether nothing follows the ops of this call: no compiler or tracer, no dispatch or function mode, no functorch transform, no
    profiler (whose record names them).  Never where that cannot be told."""
    if torch.compiler.is_compiling() or _FOLLOWERS is None:
        return False
    dispatch_modes, function_modes, transform, tracing, profiling, _ = _FOLLOWERS
    return not (dispatch_modes() > 0 or function_modes() > 0 or transform() is not None or tracing() or profiling())


def call(op, *args):
    """``op(*args)``: the registered function itself in a plain eager call on real tensors, without a gradient to record.  Tensor
    subclasses, tensors on the meta device and those whose memory is not their value (negative views, such as the imaginary part of a
    conjugate, and autograd's zero tensors, which have none) go through the op, whose dispatcher layers know what to do with them.  So
    does what autograd would record, also in a backward that is recorded itself (``create_graph=True``): the op knows its formula, or
    that it has none and a second derivative must raise."""
    if not plain_eager():
        return op(*args)
    grad = torch.is_grad_enabled()
    for a in args:
        if isinstance(a, torch.Tensor) and (type(a) not in _PLAIN or a.is_meta or (grad and a.requires_grad) or a.is_neg()
                                            or a._is_zerotensor()):
            return op(*args)
    return op.eager(*args)


def device_guard(dev: torch.device):
    """Makes ``dev`` the current device for a ``with`` block."""
    return _NO_GUARD if torch.cuda.current_device() == dev.index else torch.cuda.device(dev)


def raw_stream(dev: torch.device) -> int:
    """The current stream of ``dev`` as the integer the C ABI takes."""
    if _raw_stream is None:
        return torch.cuda.current_stream(dev).cuda_stream
    return _raw_stream(torch.cuda.current_device() if dev.index is None else dev.index)
