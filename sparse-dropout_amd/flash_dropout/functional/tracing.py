"""The compiled functions under ``torch.jit.trace``.

A trace records operators and Python autograd functions.  The native functions are neither: of a call into them it would
record the allocation of the result and nothing that fills it, and the traced program would return uninitialised memory.
So while a trace is being taken their call is made inside a Python autograd function, which the trace records as one
operation on the call's tensors and runs again whenever the traced program runs.
"""
from __future__ import annotations

import functools
from collections.abc import Iterable

import torch

_is_tracing = torch._C._is_tracing  # what torch.jit.is_tracing asks outside of a script, in half of its time


class _Slot(int):
    """The place of a tensor among the operation's inputs."""


def _take(value, tensors: list):
    """``value`` with every tensor moved to ``tensors`` and a slot in its place."""
    if isinstance(value, torch.Tensor):
        tensors.append(value)
        return _Slot(len(tensors) - 1)
    if isinstance(value, Iterable) and not isinstance(value, str):
        return [_take(v, tensors) for v in value]
    return value


def _put(value, tensors):
    if isinstance(value, _Slot):
        return tensors[value]
    return [_put(v, tensors) for v in value] if isinstance(value, list) else value


class _RecordedCall(torch.autograd.Function):
    @staticmethod
    def forward(ctx, call, *tensors):
        ctx.leaves = [t.detach().requires_grad_(need) for t, need in zip(tensors, ctx.needs_input_grad[1:])]
        with torch.enable_grad(), torch.autocast("cuda", enabled=False):
            ctx.result = call(ctx.leaves)
        return ctx.result.detach()

    @staticmethod
    def backward(ctx, grad):
        ctx.saved_tensors  # (raises once the graph was freed)
        wanted = [t for t in ctx.leaves if t.requires_grad]
        # retained: whether there will be another backward is the outer graph's to say
        grads = iter(torch.autograd.grad(ctx.result, wanted, grad, retain_graph=True))
        return (None, *(next(grads) if t.requires_grad else None for t in ctx.leaves))


def traceable(function):
    """Makes a function of tensors that calls native code one recorded operation under ``torch.jit.trace``."""

    @functools.wraps(function)
    def run(*args, **kwargs):
        if not _is_tracing():
            return function(*args, **kwargs)
        tensors: list[torch.Tensor] = []
        names, values = list(kwargs), _take([*args, *kwargs.values()], tensors)
        if torch.is_autocast_enabled("cuda"):  # the casts are the trace's own
            dtype = torch.get_autocast_dtype("cuda")
            tensors = [t.to(dtype) if t.is_floating_point() else t for t in tensors]

        def call(given):
            filled = _put(values, given)
            return function(*filled[:len(args)], **dict(zip(names, filled[len(args):])))

        return _RecordedCall.apply(call, *tensors)

    return run
