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

_TYPES = (torch.Tensor, torch.nn.Parameter)


def _torch_state():
    """What ``plain`` reads of torch, which has no public way to ask for it: (keys of a tensor,
    keys that this thread adds to a call, function modes active, profiler active, forward-mode
    level, the keys of an ordinary GPU tensor, those of a thread with no mode active)."""
    key, key_set = torch._C.DispatchKey, torch._C.DispatchKeySet
    # an ordinary GPU tensor (an inference tensor has no autograd keys) ...
    inference = key_set(key.CUDA).add(key.AutocastCUDA)
    tensor_keys = frozenset((
        inference.raw_repr(), inference.add(key.AutogradCUDA).add(key.ADInplaceOrView).raw_repr()))
    # ... and what a thread adds to every call when no mode is active (in inference mode, and
    # otherwise): the Python modes, functorch's transforms, functionalization and tracing add theirs
    thread_keys = frozenset((
        key_set(key.BackendSelect).raw_repr(),
        key_set(key.BackendSelect).add(key.ADInplaceOrView).raw_repr()))
    state = (torch._C._dispatch_keys, torch._C._dispatch_tls_local_include_set,
             torch._C._len_torch_function_stack, torch.autograd._profiler_enabled,
             lambda: _fwd_ad._current_level, tensor_keys, thread_keys)
    for read in (*state[1:5], lambda: state[0](torch.empty(0)).raw_repr(),
                 lambda: state[1]().raw_repr()):
        read()
    return state


try:
    _STATE = _torch_state()
except (AttributeError, TypeError, RuntimeError):   # a torch that keeps this elsewhere: every call takes the general route
    _STATE = None


def plain(*args) -> bool:
    """Whether a call on these arguments has nothing to record, trace, transform, wrap or
    profile: then the dispatcher would end in the op's body with the same arguments."""
    if torch.compiler.is_compiling() or _STATE is None:
        return False
    keys_of, thread_keys_now, function_modes, profiling, _, tensor_keys, thread_keys = _STATE
    if (profiling() or function_modes() != 0
            or thread_keys_now().raw_repr() not in thread_keys):
        return False
    grad = torch.is_grad_enabled()
    for t in args:
        if type(t) in _TYPES:
            if keys_of(t).raw_repr() not in tensor_keys or (grad and t.requires_grad):
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
    if (torch.compiler.is_compiling() or torch.is_grad_enabled() or not plain(*args)
            or _STATE[4]() >= 0):
        return function.apply(*args)
    out = function.forward(NoGraph(), *args)
    # (an input that comes back as an output is a view of it, as from apply)
    if isinstance(out, tuple):
        return tuple(o.view_as(o) if any(o is a for a in args) and isinstance(o, torch.Tensor)
                     else o for o in out)
    return out.view_as(out) if any(out is a for a in args) else out
