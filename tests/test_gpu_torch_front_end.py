"""The torch front end's host path on real kernels: what a call under a trace, in a gradient or beside other threads does."""

import threading
import time

import pytest
import torch
import torch.autograd.forward_ad as fwAD

import gpu_ragged_dot_amd as rd
from gpu_ragged_dot_amd import _capi, moe, ops
from gpu_ragged_dot_amd._native import lib as _native

pytestmark = pytest.mark.gpu


def _layer_inputs(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rand = lambda *s: torch.randn(s, generator=gen, device="cuda").to(torch.bfloat16).requires_grad_()
    return rand(40, 64), rand(5, 64, 96), rand(5, 96, 64), torch.rand((40, 2), generator=gen, device="cuda").requires_grad_(), \
        torch.randint(5, (40, 2), generator=gen, device="cuda", dtype=torch.int32)


def _layer(h, w_in, w_out, weights, ids):
    r = moe.route(ids, 5)
    hidden = torch.nn.functional.silu(rd.ragged_dot(moe.dispatch(h, r), w_in, r.group_sizes))
    return moe.combine(rd.ragged_dot(hidden, w_out, r.group_sizes), r, weights)


def test_a_traced_layer_runs_its_kernels():
    """The traced layer gives the eager one's bits and gradients, on other inputs than the recorded ones."""
    print("traced layer", flush=True)
    traced = torch.jit.trace(_layer, _layer_inputs(0), check_trace=False)
    for seed in (1, 2):
        args = _layer_inputs(seed)
        want, got = _layer(*args), traced(*args)
        assert torch.equal(got, want)
        dout = torch.randn_like(want)
        for a, b in zip(*(torch.autograd.grad(y, args[:4], dout) for y in (got, want))):
            assert torch.equal(a, b)
    with torch.no_grad():
        assert torch.equal(traced(*args), want)


def test_a_traced_transposed_product_runs_its_kernel():
    print("traced tgmm", flush=True)
    gs = torch.tensor([5, 0, 11], dtype=torch.int32, device="cuda")
    rand = lambda n: torch.randn((16, n), device="cuda").to(torch.bfloat16).requires_grad_()
    call = lambda x, y: rd.tgmm(x, y, gs)
    traced = torch.jit.trace(call, (rand(32), rand(24)), check_trace=False)
    args = rand(32), rand(24)
    want, got = call(*args), traced(*args)
    assert torch.equal(got, want)
    for a, b in zip(*(torch.autograd.grad(y, args, torch.ones_like(want)) for y in (got, want))):
        assert torch.equal(a, b)


HP = dict(block_m=64, block_k=64, block_n=64, interpret=False, compute_dtype=None, acc_dtype=torch.float32, chunk_m=512)


def test_a_plan_for_the_product_leaves_its_gradients_to_the_library():
    """float32, contractions that are cut along K by default: a plan that forbids the cut holds for the product it is given to."""
    gs = torch.tensor([70, 0, 130], dtype=torch.int32, device="cuda")
    vid = [v.id for v in _capi.variants() if v.name.decode().startswith("fr64x64")][0]
    plan = _capi.Plan(vid, split_k=-1)
    for call, default, shapes in (
            (lambda x, A: ops._gmm(x, A, gs, **HP, trans_rhs=False, plan=plan), lambda x, A: rd.gmm(x, A, gs), ((200, 192), (3, 192, 2048))),
            (lambda x, y: ops._tgmm(x, y, gs, **HP, plan=plan), lambda x, y: rd.tgmm(x, y, gs), ((200, 192), (200, 2048)))):
        print(f"gradients beside a plan, {shapes}", flush=True)
        args = [torch.randn(*s, device="cuda", requires_grad=True) for s in shapes]
        out = call(*args)
        dout = torch.randn_like(out)
        got, want = (torch.autograd.grad(y, args, dout) for y in (out, default(*args)))
        uncut = ops._gmm_fwd(*((dout, args[1]) if out.dim() == 2 else (args[1], dout)), gs, **HP, trans_rhs=True, plan=plan)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        assert not torch.equal(got[0], uncut)


@pytest.mark.parametrize("op", ["gmm", "tgmm"])
def test_an_error_in_a_gradient_keeps_its_type(op):
    """A gradient whose plan names no tile shape: refused on the host, with the error a product of its own raises."""
    gs = torch.tensor([3, 5], dtype=torch.int32, device="cuda")
    rand = lambda *s: torch.randn(*s, device="cuda").to(torch.bfloat16).requires_grad_()
    x, other = rand(8, 64), rand(2, 64, 64) if op == "gmm" else rand(8, 64)
    good, bad = (-1, 0, 0, 0, 0), (10 ** 6, 0, 0, 0, 0)
    for plans, wanted in (((good, bad, good), x), ((good, good, bad), other)):
        print(f"failing gradient of {op}", flush=True)
        if op == "gmm":
            out = _native.gmm(x, other, gs, False, _capi.RD_DTYPE_BF16, -1, plans)
        else:
            out = _native.tgmm(x, other, gs, _capi.RD_DTYPE_BF16, -1, -1, plans)
        with pytest.raises(_capi.RaggedDotError, match="out of range") as e:
            torch.autograd.grad(out, wanted, torch.ones_like(out))
        assert e.value.status == _capi.RD_ERR_INVALID_ARGUMENT


def test_a_cotangent_with_a_forward_mode_tangent_is_refused():
    """The gradient of a gradient along a direction is not implemented: an answer without a tangent would read as zero."""
    args = _layer_inputs(3)
    r = moe.route(args[4], 5)
    y = torch.randn(80, 64, device="cuda").requires_grad_()
    outs = {"gmm": (rd.gmm(moe.dispatch(args[0].detach(), r), args[1], r.group_sizes), args[1]), "dispatch": (moe.dispatch(args[0], r), args[0]),
            "tgmm": (rd.tgmm(y, y.detach(), r.group_sizes), y), "combine": (moe.combine(y, r, args[3]), y)}
    for name, (out, wanted) in outs.items():
        print(f"dual cotangent of {name}", flush=True)
        with fwAD.dual_level(), pytest.raises(NotImplementedError, match="forward-mode"):
            torch.autograd.grad(out, wanted, fwAD.make_dual(torch.ones_like(out), torch.ones_like(out)))


@pytest.mark.parametrize("op", ["gmm", "tgmm"])
def test_other_threads_run_while_a_call_waits_for_the_device(op):
    """A copy from host memory waits for the stream: other Python threads must not wait with it."""
    print(f"waiting {op}", flush=True)
    x, A = torch.randn(16, 64, device="cuda").bfloat16(), torch.randn(2, 64, 64, device="cuda").bfloat16()
    y, sizes = torch.randn(16, 64, device="cuda").bfloat16(), torch.tensor([9, 7])  # int64 on the host
    call = {"gmm": lambda: rd.gmm(x, A, sizes), "tgmm": lambda: rd.tgmm(x, y, sizes)}[op]
    call()
    big = torch.randn(8192, 8192, device="cuda")
    big @ big
    torch.cuda.synchronize()
    ticks, done = [0], threading.Event()

    def tick():
        while not done.wait(0.001):
            ticks[0] += 1

    other = threading.Thread(target=tick)
    for _ in range(30):
        big @ big  # 10 ms each and more
    other.start()
    before, start = ticks[0], time.perf_counter()
    call()
    waited, passed = time.perf_counter() - start, ticks[0] - before
    done.set()
    other.join()
    torch.cuda.synchronize()
    assert waited > 0.05, "the call was meant to wait"
    assert passed > 100 * waited, f"{passed} ticks of a millisecond in {waited:.3f} s"


@pytest.mark.parametrize("trans_rhs", [False, True])
def test_a_small_product_at_an_odd_address_needs_little_memory(trans_rhs):
    print(f"odd address, trans_rhs {trans_rhs}", flush=True)
    gs = torch.tensor([20, 0, 30, 14], dtype=torch.int32, device="cuda")
    A = torch.randn(4, 64, 64, device="cuda").bfloat16()
    aligned = torch.randn(64, 64, device="cuda").bfloat16()
    x = torch.empty(64 * 64 + 1, dtype=torch.bfloat16, device="cuda")[1:].view(64, 64).copy_(aligned)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    y = rd.gmm(x, A, gs, trans_rhs=trans_rhs)
    assert torch.cuda.max_memory_allocated() - before < 1 << 20
    ref = rd.gmm(aligned.float(), A.float(), gs, trans_rhs=trans_rhs)
    assert torch.linalg.norm(y.float() - ref) <= 2.0 ** -8 * torch.linalg.norm(ref)  # one rounding to bfloat16


def test_routing_arrays_that_the_kernels_cannot_read_are_refused():
    """Host memory and arrays shorter than the routing says are refused on the host: no kernel sees their addresses."""
    ids = torch.randint(4, (16, 2), device="cuda", dtype=torch.int32)
    r = moe.route(ids, 4)
    h, y = torch.randn(16, 8, device="cuda"), torch.randn(32, 8, device="cuda")
    w = torch.rand(16, 2, device="cuda")
    for message, call in (
            ("same device", lambda: moe.combine(y, r, w.cpu())),
            ("same device", lambda: moe.combine(y, r._replace(row_of_slot=r.row_of_slot.cpu()), w)),
            ("same device", lambda: moe.dispatch(h, r._replace(row_of_slot=r.row_of_slot.cpu()))),
            ("same device", lambda: moe.dispatch(h, r._replace(slot_of_row=r.slot_of_row.cpu()))),
            ("same device", lambda: moe._dispatch(h, r, w.cpu().reshape(-1))),
            ("32 slots", lambda: moe._dispatch(h, r, w[:8].reshape(-1))),
            ("32 slots", lambda: moe.dispatch(h, r._replace(slot_of_row=r.slot_of_row[:8]))),
            ("32 slots", lambda: moe.combine(y, r._replace(row_of_slot=r.row_of_slot.view(16, 2)[:, 0].repeat(1)), w))):
        with pytest.raises((RuntimeError, ValueError), match=message):
            call()
    assert moe.combine(moe.dispatch(h, r), r, w).shape == h.shape
