"""The routing kernels at the edges of their dispatch, against the oracle: one slot fewer and more than a block ranks, than
the one-kernel form takes and than the two-kernel form takes; as many experts as their tables hold and one more; dropped
slots; every element type of the gradient of the combine weights with row lengths on and off 16 bytes; matrices larger
than the last-level cache, which are read past it."""

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import moe
from oracle import moe_glue_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [1, 63, 64, 1023, 1024, 1025, 16 * 1024 - 1, 16 * 1024, 16 * 1024 + 1, 64 * 1024, 64 * 1024 + 1])
@pytest.mark.parametrize("g,drop", [(1, 0.0), (8, 0.1), (128, 0.0), (512, 0.3), (513, 0.0)])
def test_route_edges(slots, g, drop):
    print(f"route slots {slots} g {g} drop {drop}", flush=True)
    rng = np.random.default_rng(slots + g)
    ids = rng.integers(0, g, size=(slots, 1)).astype(np.int32)
    ids[rng.random((slots, 1)) < drop] = g if g % 2 else -1
    r = moe.route(torch.from_numpy(ids).cuda(), g)
    sizes, row_of_slot, slot_of_row = moe_glue_oracle.route(ids, g)
    assert np.array_equal(r.group_sizes.cpu().numpy(), sizes)
    assert np.array_equal(r.row_of_slot.cpu().numpy(), row_of_slot)
    assert np.array_equal(r.slot_of_row.cpu().numpy(), slot_of_row)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("top_k,d", [(1, 8), (4, 512), (5, 520), (8, 7), (17, 1032), (64, 72)])
def test_combine_and_weight_gradient(top_k, d, dtype):
    print(f"combine top_k {top_k} d {d} {dtype}", flush=True)
    tokens, g = 33, 70
    rng = np.random.default_rng(top_k * d)
    ids = np.stack([rng.permutation(g)[:top_k] for _ in range(tokens)]).astype(np.int32)
    ids[rng.random(ids.shape) < 0.1] = -1
    r = moe.route(torch.from_numpy(ids).cuda(), g)
    y = torch.randn(tokens * top_k, d, device="cuda").to(dtype).requires_grad_()
    w = torch.rand(tokens, top_k, device="cuda").requires_grad_()
    dout = torch.randn(tokens, d, device="cuda").to(dtype)
    out = moe.combine(y, r, w)
    dw = torch.autograd.grad(out, w, dout)[0].reshape(-1).double().cpu().numpy()
    row = r.row_of_slot.cpu().numpy()
    yv, gv, wv = (t.detach().double().cpu().numpy() for t in (y, dout, w))
    live = (row >= 0).reshape(tokens, top_k)
    picked = yv[np.maximum(row, 0)].reshape(tokens, top_k, d) * live[..., None]
    # fp32 sums of d (dw) or top_k (out) products: at most that many roundings of 2^-24 of the sum of magnitudes; out is
    # rounded once more to its type
    dw_ref, dw_mag = np.einsum("tsd,td->ts", picked, gv), np.einsum("tsd,td->ts", np.abs(picked), np.abs(gv))
    assert np.all(np.abs(dw.reshape(tokens, top_k) - dw_ref) <= (d + 8) * 2.0 ** -24 * dw_mag)
    half_ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[dtype]
    ref, mag = np.einsum("tsd,ts->td", picked, wv), np.einsum("tsd,ts->td", np.abs(picked), wv)
    got = out.detach().double().cpu().numpy()
    assert np.all(np.abs(got - ref) <= half_ulp * np.abs(ref) + (top_k + 1) * 2.0 ** -24 * mag + 2.0 ** -24)


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 8200), (torch.float16, 8200), (torch.float32, 4100)], ids=["bf16", "f16", "f32"])
def test_rows_beyond_the_last_level_cache(dtype, d):
    """More than 256 MiB of rows: the same bits as two calls of half the size, which read through the caches."""
    print(f"rows beyond the cache {dtype}", flush=True)
    half, top_k, g = 4099, 2, 5
    y = torch.randn(2 * half * top_k, d, device="cuda").to(dtype)
    assert y.numel() * y.element_size() > 256 << 20 > y.numel() * y.element_size() // 2
    r = moe.route(torch.randint(-1, g, (2 * half, top_k), device="cuda", dtype=torch.int32), g)
    w = torch.rand(2 * half, top_k, device="cuda").requires_grad_()
    dout = torch.randn(2 * half, d, device="cuda").to(dtype)
    out = moe.combine(y, r, w)
    dw, = torch.autograd.grad(out, w, dout)
    slots = torch.arange(half * top_k, device="cuda", dtype=torch.int32)
    for part in (slice(0, half), slice(half, 2 * half)):
        rows = r.row_of_slot.view(-1, top_k)[part].reshape(-1)
        own = moe.Routing(r.group_sizes, torch.where(rows < 0, rows, slots), slots, half, top_k)
        w_part = w.detach()[part].clone().requires_grad_()
        out_part = moe.combine(y[rows.clamp(min=0).long()], own, w_part)
        dw_part, = torch.autograd.grad(out_part, w_part, dout[part])
        assert torch.equal(out[part], out_part) and torch.equal(dw[part], dw_part)
    assert not dw.view(-1)[r.row_of_slot < 0].any() and dw.any()


def test_dispatch_gradient_twice():
    """A dispatch keeps no operand for its gradient, so asking for it twice needs no retain_graph."""
    ids = torch.tensor([[0, 1], [2, 0], [1, 1]], device="cuda")
    r = moe.route(ids, 3)
    h = torch.randn(3, 16, device="cuda").requires_grad_()
    x = moe.dispatch(h, r)
    dx = torch.randn_like(x)
    first, again = (torch.autograd.grad(x, h, dx)[0] for _ in range(2))
    assert torch.equal(first, again)
