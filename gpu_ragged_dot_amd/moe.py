"""Token routing around ``ragged_dot`` for a mixture of experts, on the device.

``ragged_dot`` takes rows sorted by group; the reference leaves producing them to its caller (its tests build sorted
rows directly, tests.py:51-71).  This module is that caller's side, each function one call across the C ABI
(``rd_moe_*`` in ``include/ragged_dot_hip.h``):

    routing = route(expert_ids, num_groups)                 # group_sizes, row_of_slot, slot_of_row
    x = dispatch(h, routing)                                # [tokens * top_k, d], rows sorted by expert
    y = ragged_dot(x, W, routing.group_sizes)               # the op itself
    out = combine(y, routing, weights)                      # [tokens, n]

``dispatch`` and ``combine`` are differentiable (each one's backward is the other kernel; the gradient of the combine
weights is ``rd_moe_combine_wgrad``).  torch supplies device memory, the stream and the autograd engine; the host side of
each call is native (``csrc/rd_torch.cpp``).
"""

from __future__ import annotations

from typing import NamedTuple, Optional

import torch

from . import _tracing
from ._native import lib as _native

__all__ = ["Routing", "route", "dispatch", "combine"]


class Routing(NamedTuple):
    group_sizes: torch.Tensor   # int32 [g]      rows per expert
    row_of_slot: torch.Tensor   # int32 [tokens * top_k]  row of the sorted matrix each (token, choice) went to, -1 = dropped
    slot_of_row: torch.Tensor   # int32 [tokens * top_k]  inverse; -1 for rows past sum(group_sizes)
    tokens: int
    top_k: int


def route(expert_ids: torch.Tensor, num_groups: int) -> Routing:
    """Stable counting sort of the (token, choice) pairs by expert id.  ``expert_ids`` is integer ``[tokens, top_k]``;
    ids outside ``[0, num_groups)`` mark dropped pairs."""
    if _tracing.active():
        outs = _tracing.record(lambda ids: _native.moe_route(ids, num_groups), expert_ids)
        return Routing(*outs, *map(int, expert_ids.shape))
    group_sizes, row_of_slot, slot_of_row = _native.moe_route(expert_ids, num_groups)
    return Routing(group_sizes, row_of_slot, slot_of_row, *expert_ids.shape)


def _dispatch(h, r: Routing, row_scale):
    """The kernel alone (no autograd node); ``row_scale``: a float32 factor per slot, or None."""
    return _native.moe_dispatch_rows(h, row_scale, r.row_of_slot, r.slot_of_row, r.tokens, r.top_k)


def _combine(y, r: Routing, weights):
    """The kernel alone (no autograd node)."""
    with torch.no_grad():
        return _native.moe_combine(y, weights, r.row_of_slot, r.slot_of_row, r.tokens, r.top_k)


def dispatch(h: torch.Tensor, routing: Routing) -> torch.Tensor:
    """``x[row] = h[token of row]``: ``[tokens, d] -> [tokens * top_k, d]`` sorted by expert; rows past
    ``sum(group_sizes)`` are zero."""
    if _tracing.active():
        return _tracing.record(lambda *t: dispatch(t[0], routing._replace(row_of_slot=t[1], slot_of_row=t[2])),
                               h, routing.row_of_slot, routing.slot_of_row)
    return _native.moe_dispatch(h, routing.row_of_slot, routing.slot_of_row, routing.tokens, routing.top_k)


def combine(y: torch.Tensor, routing: Routing, weights: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``out[token] = sum_choice weights[token, choice] * y[row of (token, choice)]`` with fp32 accumulation;
    ``weights`` is ``[tokens, top_k]`` (None = 1)."""
    if _tracing.active():
        return _tracing.record(lambda *t: combine(t[0], routing._replace(row_of_slot=t[1], slot_of_row=t[2]), *t[3:]),
                               y, routing.row_of_slot, routing.slot_of_row, *(() if weights is None else (weights,)))
    return _native.moe_combine(y, weights, routing.row_of_slot, routing.slot_of_row, routing.tokens, routing.top_k)
