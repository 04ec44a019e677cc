"""The work that users of this package have it do, as cases that a timing program can prepare, run and compare.

A case is one pass of one of these kinds through the public entry points (``ragged_dot`` and its gradients, ``moe.route``
/ ``dispatch`` / ``combine``):

* ``forward``    one ragged product, as in serving;
* ``train``      the product and, through autograd, the gradients of both operands;
* ``moe_serve``  a mixture-of-experts layer: route, dispatch, product, SiLU, product, combine;
* ``moe_train``  the same layer with the gradients of its input, its two weight tensors and its combine weights.

Sizes are those of this repository's workloads, benchmark, tuner and tests, or generic ones around them.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import gpu_ragged_dot_amd as rd

_TYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32, "f8": torch.float8_e4m3fn}
_BYTES = {"bf16": 2, "f16": 2, "f32": 4, "f8": 1}


def _product(kind, m, k, n, g, dtype="bf16", compute="same", trans_rhs=False, routing="topk", fill=1.0, **name):
    """A ragged product over ``m`` rows.  ``routing`` says how the rows fall on the groups, ``fill`` which share of the m
    rows belongs to a group at all (a padded batch has a tail of rows that do not)."""
    return dict(kind=kind, m=m, k=k, n=n, g=g, dtype=dtype, compute=compute, trans_rhs=trans_rhs, routing=routing,
                fill=fill, **name)


def _layer(kind, tokens, top_k, d, f, g, dtype="bf16", **name):
    """A mixture-of-experts layer of ``g`` experts d -> f -> d, ``top_k`` of them for each token."""
    return dict(kind=kind, tokens=tokens, top_k=top_k, d=d, f=f, g=g, dtype=dtype, **name)


def listed():
    return [
        # one decoding step of 8 sequences, top-8 of 128 experts: the smallest call in serving, a stream over the weights
        _product("forward", 64, 2048, 768, 128, name="decode_8_tokens"),
        # a batch of 64 sequences on weights stored [g, n, k], as checkpoints hold them
        _product("forward", 512, 2048, 768, 128, trans_rhs=True, name="decode_64_tokens_transposed"),
        # a whole layer for a serving batch of 256 tokens in float16
        _layer("moe_serve", 256, 8, 2048, 768, 128, dtype="f16", name="moe_layer_256_tokens"),
        # the smallest training call: unit-test and toy sizes, where launches and the host's work count
        _product("train", 512, 256, 512, 4, name="train_tiny"),
        # prompt processing with quantised weights and activations
        _product("forward", 16384, 4096, 14336, 8, dtype="f8", name="prefill_float8"),
        # float32 training
        _product("train", 8192, 2048, 2048, 16, dtype="f32", routing="softmax", name="train_float32"),
        # float32 arrays multiplied in bfloat16 (compute_dtype), the usual mixed precision
        _product("train", 8192, 4096, 4096, 8, dtype="f32", compute="bf16", name="train_float32_compute_bf16"),
        # row pitches that are no multiple of 16 bytes, a padded batch
        _product("train", 4099, 1001, 1515, 12, routing="softmax", fill=0.9, name="train_odd_sizes"),
        # the shape the reference tunes for, with its softmax-distributed groups
        _product("train", 8192, 7168, 2048, 32, routing="softmax", name="train_32_groups"),
        # a training step's expert layer: 4096 tokens, top-8 of 128 experts
        _layer("moe_train", 4096, 8, 2048, 768, 128, name="moe_layer_train"),
        # many rows per expert: the matrix cores are what bounds it
        _product("train", 16384, 4096, 14336, 8, name="train_8_large_experts"),
        # few rows per expert, skewed, a tenth of the experts without any: memory is what bounds it
        _product("train", 32768, 7168, 2048, 256, routing="zipf", name="train_256_skewed_experts"),
    ]


def _log_int(rng, lo, hi, step=1):
    """An integer in [lo, hi], uniform in its logarithm, rounded to a multiple of ``step``."""
    return max(lo, min(hi, step * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)))


def _affordable(case):
    """No costlier than the largest listed cases (about 5 ms a pass), with three states on one card."""
    w = work(case)
    d1, d2 = (case["d"], 2 * case["f"]) if "tokens" in case else (case["k"], case["n"])
    if case["g"] * d1 * d2 * _BYTES[case["dtype"]] > 16e9:
        return False
    rate = {"f32": 8e13, "f8": 1e15}.get(case["dtype"], 1e15)
    if case.get("compute") == "bf16":
        rate = 3e14
    elif "k" in case and case["dtype"] != "f32" and (case["k"] % 8 or case["n"] % 8):
        rate = 8e13
    return w["flops"] / rate < 4e-3 and w["bytes"] < 16e9


def draw(rng):
    while True:
        kind = rng.choice(["decode", "decode", "forward", "train", "train", "train", "moe_serve", "moe_train"])
        if kind in ("moe_serve", "moe_train"):
            serve = kind == "moe_serve"
            g = rng.choice([8, 16, 32, 64, 128, 256])
            case = _layer(kind, _log_int(rng, 16, 1024) if serve else _log_int(rng, 512, 8192), rng.randint(1, 8),
                          _log_int(rng, 512, 7168, 64), _log_int(rng, 256, 4096, 64), g,
                          dtype=rng.choice(["bf16", "bf16", "f16"]))
        elif kind == "decode":
            g = _log_int(rng, 8, 256)
            case = _product("forward", rng.randint(1, 8) * _log_int(rng, 1, 128), _log_int(rng, 512, 8192, 64),
                            _log_int(rng, 256, 8192, 64), g, dtype=rng.choice(["bf16", "bf16", "f16", "f8"]),
                            trans_rhs=rng.random() < 0.5)
        else:
            types = ["bf16", "bf16", "f16", "f8"] if kind == "forward" else ["bf16", "bf16", "bf16", "f16", "f32", "f32"]
            dtype = rng.choice(types)
            odd = dtype != "f8" and rng.random() < 0.2
            k, n = (_log_int(rng, 57, 4096) if odd else _log_int(rng, 256, 16384, 16) for _ in range(2))
            case = _product(kind, _log_int(rng, 256, 32768), k, n, _log_int(rng, 2, 256), dtype=dtype,
                            compute="bf16" if dtype == "f32" and rng.random() < 0.5 else "same",
                            trans_rhs=rng.random() < 0.3, routing=rng.choice(["topk", "softmax", "zipf"]),
                            fill=rng.choice([1.0, 1.0, 0.8]))
        if _affordable(case):
            return case


def _rows(case):
    return round(case["m"] * case["fill"])


def _shares(routing, g, rng):
    """The probability of each group: equal experts, softmax of N(0, 1) logits as the tuner's sizes, or a permuted
    Zipf law with a tenth of the groups empty."""
    if routing == "softmax":
        p = np.exp(rng.standard_normal(g))
    elif routing == "zipf":
        p = (rng.permutation(g) + 1.0) ** -1.1
        p[rng.choice(g, size=g // 10, replace=False)] = 0.0
    else:
        p = np.ones(g)
    return p / p.sum()


def _normal(gen, shape, dtype, scale=1.0):
    """N(0, scale^2) on the GPU, in slabs along the first axis so that staging stays small beside a large tensor."""
    staged = torch.bfloat16 if dtype == torch.bfloat16 else torch.float16 if dtype == torch.float16 else torch.float32
    out = torch.empty(shape, dtype=dtype, device="cuda")
    for part in out.split(max(1, shape[0] // 8)):
        part.copy_(torch.randn(part.shape, generator=gen, device="cuda", dtype=staged).mul_(scale))
    return out


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rng = np.random.default_rng(seed)
    dtype, g = _TYPES[case["dtype"]], case["g"]
    if "tokens" in case:
        tokens, d, f, train = case["tokens"], case["d"], case["f"], case["kind"] == "moe_train"
        logits = torch.randn((tokens, g), generator=gen, device="cuda")
        best, ids = logits.topk(case["top_k"], dim=1)
        state = dict(case=case, ids=ids.to(torch.int32), weights=best.softmax(dim=1),
                     h=_normal(gen, (tokens, d), dtype), w_in=_normal(gen, (g, d, f), dtype, d ** -0.5),
                     w_out=_normal(gen, (g, f, d), dtype, f ** -0.5))
        if train:
            state["dout"] = _normal(gen, (tokens, d), dtype)
            for key in ("h", "w_in", "w_out", "weights"):
                state[key].requires_grad_()
        return state
    m, k, n = case["m"], case["k"], case["n"]
    sizes = rng.multinomial(_rows(case), _shares(case["routing"], g, rng)).astype(np.int32)
    # quantised weights span the range of their type (their scales are applied outside the product)
    scale = 1.0 if case["dtype"] == "f8" else k ** -0.5
    state = dict(case=case, sizes=torch.from_numpy(sizes).cuda(), x=_normal(gen, (m, k), dtype),
                 w=_normal(gen, (g, n, k) if case["trans_rhs"] else (g, k, n), dtype, scale))
    if case["kind"] == "train":
        state["dy"] = _normal(gen, (m, n), dtype)
        state["x"].requires_grad_()
        state["w"].requires_grad_()
    return state


def _expert_layer(s):
    routing = rd.moe.route(s["ids"], s["case"]["g"])
    rows = rd.moe.dispatch(s["h"], routing)
    hidden = torch.nn.functional.silu(rd.ragged_dot(rows, s["w_in"], routing.group_sizes))
    return rd.moe.combine(rd.ragged_dot(hidden, s["w_out"], routing.group_sizes), routing, s["weights"])


def run(s):
    case = s["case"]
    if case["kind"] == "moe_serve":
        with torch.no_grad():
            return _expert_layer(s)
    if case["kind"] == "moe_train":
        out = _expert_layer(s)
        grads = torch.autograd.grad(out, (s["h"], s["w_in"], s["w_out"], s["weights"]), s["dout"])
        return (out.detach(),) + grads
    compute = torch.bfloat16 if case["compute"] == "bf16" else None
    y = rd.ragged_dot(s["x"], s["w"], s["sizes"], trans_rhs=case["trans_rhs"], compute_dtype=compute)
    if case["kind"] == "forward":
        return y
    return (y.detach(),) + torch.autograd.grad(y, (s["x"], s["w"]), s["dy"])


def _groups_with_rows(rows, p):
    """How many groups get a row at all, on average."""
    return float((1.0 - (1.0 - p) ** rows).sum())


def work(case):
    e, g = _BYTES[case["dtype"]], case["g"]
    if "tokens" in case:
        tokens, d, f, slots = case["tokens"], case["d"], case["f"], case["tokens"] * case["top_k"]
        live = g * (1.0 - (1.0 - case["top_k"] / g) ** tokens)
        moved = 2 * tokens * d * e + 2 * live * d * f * e + 8 * slots
        flops = 4.0 * slots * d * f
        if case["kind"] == "moe_train":
            return {"bytes": moved + 2 * tokens * d * e + 2 * g * d * f * e + 4 * slots, "flops": 3 * flops}
        return {"bytes": moved, "flops": flops}
    m, k, n, rows = case["m"], case["k"], case["n"], _rows(case)
    live = _groups_with_rows(rows, _shares(case["routing"], g, np.random.default_rng(0)))
    out = 2 if case["dtype"] == "f8" else e
    moved = rows * k * e + live * k * n * e + m * n * out + 4 * g
    flops = 2.0 * rows * k * n
    if case["kind"] == "train":
        return {"bytes": moved + rows * n * e + m * k * e + g * k * n * e, "flops": 3 * flops}
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """Four times the distance to the same products summed in float64 and rounded once per step of the path, over the
    listed cases and two dozen drawn ones: float32 sums 2e-6 (largest single difference 3e-5), whether or not the
    operands are rounded to bfloat16 first; float16 outputs 7e-5 (2e-3); bfloat16 outputs 2.5e-4 through a whole layer,
    5.6e-4 for a single row of float8 products (1.5e-2: two units in the last place)."""
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 1e-4}
    if case["dtype"] == "f16":
        return {"rel": 3e-4, "max": 8e-3}
    return {"rel": 2e-3, "max": 6e-2}
