"""Calls of the native front end under ``torch.jit.trace``.

A trace records torch's own operations.  Of a native call it would see the output's allocation and nothing of the kernel, so
that the traced graph would return uninitialised memory.  A Python autograd node it records as one operation and calls again
whenever the graph runs; while a trace is recorded, every call goes through such a node.
"""

from __future__ import annotations

import threading

import torch

_tracing = torch._C._get_tracing_state
_inside = threading.local()


def active() -> bool:
    """A trace is being recorded, and not by way of a node's own forward."""
    return _tracing() is not None and not getattr(_inside, "node", False)


class _Node(torch.autograd.Function):
    """``call(*operands)`` with the native autograd nodes kept inside."""

    @staticmethod
    def forward(ctx, call, *operands):
        outer, _inside.node = getattr(_inside, "node", False), True
        try:
            with torch.enable_grad():
                ctx.operands = [t.detach().requires_grad_(need) for t, need in zip(operands, ctx.needs_input_grad[1:])]
                ctx.results = call(*ctx.operands)
            return ctx.results.detach() if isinstance(ctx.results, torch.Tensor) else tuple(t.detach() for t in ctx.results)
        finally:
            _inside.node = outer

    @staticmethod
    def backward(ctx, *grads):
        wanted = [t for t in ctx.operands if t.requires_grad]
        got = iter(torch.autograd.grad(ctx.results, wanted, grads, retain_graph=True))
        return (None, *(next(got) if t.requires_grad else None for t in ctx.operands))


record = _Node.apply
