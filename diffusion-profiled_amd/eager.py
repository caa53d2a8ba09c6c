"""What an eager call pays before its first launch.

``torch.library``'s dispatch of a Python custom op costs about as much host time as four kernel
launches, and an autograd Function's ``apply`` about two, which a sampler or an op-level program
that launches kernels of a few microseconds waits for. Where neither has anything to do -- plain
dense GPU tensors, no graph to record, nothing that traces, transforms or profiles the call --
``run`` and ``apply`` below call the op's body or the Function's forward themselves; every other
call takes the general route.

Host-bound eager calls, general route -> here: quantizing a 128x128x3x3 weight 20.3 -> 14.1 us,
a 16-image decoder block (512 -> 256 channels, 16x16, no grad) 352 -> 245 us.
"""
from __future__ import annotations

from typing import Any, Callable

import torch
from torch.autograd import forward_ad as _fwd_ad

_Key, _KeySet = torch._C.DispatchKey, torch._C.DispatchKeySet
_TYPES = (torch.Tensor, torch.nn.Parameter)
# dispatch keys of an ordinary GPU tensor (an inference tensor has no autograd keys) ...
_INFERENCE = _KeySet(_Key.CUDA).add(_Key.AutocastCUDA)
_TENSOR_KEYS = frozenset((
    _INFERENCE.raw_repr(), _INFERENCE.add(_Key.AutogradCUDA).add(_Key.ADInplaceOrView).raw_repr()))
# ... and those that a thread adds to every call when no mode is active (in inference mode, and
# otherwise): the Python modes, functorch's transforms, functionalization and tracing add theirs
_THREAD_KEYS = frozenset((
    _KeySet(_Key.BackendSelect).raw_repr(),
    _KeySet(_Key.BackendSelect).add(_Key.ADInplaceOrView).raw_repr()))


def plain(*args) -> bool:
    """Whether a call on these arguments has nothing to record, trace, transform, wrap or
    profile: then the dispatcher would end in the op's body with the same arguments."""
    if (torch.compiler.is_compiling() or torch.autograd._profiler_enabled()
            or torch._C._len_torch_function_stack() != 0
            or torch._C._dispatch_tls_local_include_set().raw_repr() not in _THREAD_KEYS):
        return False
    grad = torch.is_grad_enabled()
    for t in args:
        if type(t) in _TYPES:
            if (torch._C._dispatch_keys(t).raw_repr() not in _TENSOR_KEYS
                    or (grad and t.requires_grad)):
                return False
        elif hasattr(type(t), "__torch_function__"):    # subclasses, proxies
            return False
    return True


_BODY: dict[Any, Callable] = {}


def custom_op(name: str) -> Callable:
    """``torch.library.custom_op`` for GPU tensors that mutates nothing, known to ``run``."""
    def wrap(body: Callable):
        op = torch.library.custom_op(name, body, mutates_args=(), device_types="cuda")
        _BODY[op] = body
        return op
    return wrap


def run(op, *args):
    """``op(*args)`` of a ``custom_op`` from above."""
    return _BODY[op](*args) if plain(*args) else op(*args)


class NoGraph:
    """The context of a forward that ``apply`` calls: it records nothing, and its arguments
    were found plain (so ``run_in`` need not look at what it forms from them)."""

    def save_for_backward(self, *tensors) -> None:
        pass

    def mark_non_differentiable(self, *tensors) -> None:
        pass


def run_in(ctx, op, *args):
    """``run`` inside a Function's forward."""
    return _BODY[op](*args) if type(ctx) is NoGraph else run(op, *args)


def apply(function: type[torch.autograd.Function], *args):
    """``function.apply(*args)``; with gradients off its forward alone."""
    if (torch.compiler.is_compiling() or torch.is_grad_enabled()
            or _fwd_ad._current_level >= 0 or not plain(*args)):
        return function.apply(*args)
    out = function.forward(NoGraph(), *args)
    # (an input that comes back as an output is a view of it, as from apply)
    if isinstance(out, tuple):
        return tuple(o.view_as(o) if any(o is a for a in args) and isinstance(o, torch.Tensor)
                     else o for o in out)
    return out.view_as(out) if any(out is a for a in args) else out
