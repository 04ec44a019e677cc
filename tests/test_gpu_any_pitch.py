"""The any-pitch core (register-staged 256 x 256 and 128 x 128 tiles for odd row pitches and for float32 rounded to bf16, 128 x
128 to 64 x 64 ones for float32 as it is) and the 64 x 64 tiles that share its unaligned loads, against the oracle.

Sizes where it can go wrong: contractions of less than one slab, of one element more and less than a whole number of slabs
around the point where the pipelined loop takes over, rows of one piece only, tile edges, groups of 0, 1 and one more than
a tile's rows.  One group's operands are NaN: pieces that run past a row or a group must not carry them into the others.
"""

import numpy as np
import pytest
import torch

import gpu_ragged_dot_amd as rd
from gpu_ragged_dot_amd import _capi, ops
from oracle import ragged_dot_oracle as oracle
from tests import util

pytestmark = pytest.mark.gpu

HP = dict(block_m=64, block_k=64, block_n=64, interpret=False, acc_dtype=torch.float32, chunk_m=512)
KINDS = {_capi.RD_DTYPE_BF16: ("bfloat16", torch.bfloat16, None), _capi.RD_DTYPE_F16: ("float16", torch.float16, None),
         _capi.RD_DTYPE_F32_BF16: ("bfloat16", torch.float32, torch.bfloat16), _capi.RD_DTYPE_F32: ("float32", torch.float32, None)}
VARIANTS = [(v.id, v.name.decode(), v.dtype) for v in _capi.variants()
            if v.name.decode().startswith(("r", "hr", "cr", "cs", "fr", "s64", "h64x64", "c64"))]
# (k, n): slabs of 64 (16-bit) or 32 (float32), two of them in LDS and two in registers
SHAPES = [(8, 8), (57, 77), (63, 129), (65, 257), (191, 9), (225, 131), (257, 64), (321, 72), (385, 255), (449, 250), (577, 264)]


@pytest.mark.parametrize("vid,vname,dtype", VARIANTS, ids=[v[1] for v in VARIANTS])
@pytest.mark.parametrize("k,n", SHAPES, ids=[f"k{k}n{n}" for k, n in SHAPES])
def test_any_pitch_edges(vid, vname, dtype, k, n):
    if vname.startswith("cr") and (k % 8 or n % 8):
        k, n = (k + 7) // 8 * 8, (n + 7) // 8 * 8
    print(f"variant {vname} k {k} n {n}", flush=True)
    rounding, storage, compute = KINDS[dtype]
    gs = np.array([257, 0, 1, 63, 40, 129, 7], np.int32)
    poisoned, tail = 4, 5
    g, m, total = len(gs), int(gs.sum()) + tail, int(gs.sum())
    rng = np.random.default_rng(k * 1000 + n)
    r = lambda a: oracle.round_to(a, rounding)
    x, A, dy = r(rng.normal(size=(m, k))), r(rng.normal(size=(g, k, n)) / np.sqrt(k)), r(rng.normal(size=(m, n)))
    first = int(gs[:poisoned].sum())
    hit = slice(first, first + int(gs[poisoned]))
    clean = np.ones(m, bool)
    clean[hit] = False
    x_in, A_in, dy_in = x.copy(), A.copy(), dy.copy()
    x_in[hit], A_in[poisoned], dy_in[hit] = np.nan, np.nan, np.nan
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().to(storage)
    gs_t, plan = torch.from_numpy(gs).cuda(), _capi.Plan(vid)
    y = util.to_np(ops._gmm_fwd(dev(x_in), dev(A_in), gs_t, trans_rhs=False, compute_dtype=compute, plan=plan, **HP))
    yt = util.to_np(ops._gmm_fwd(dev(x_in), dev(np.swapaxes(A_in, 1, 2)), gs_t, trans_rhs=True, compute_dtype=compute, plan=plan, **HP))
    dA = util.to_np(ops._tgmm_fwd(dev(x_in), dev(dy_in), gs_t, compute_dtype=compute, plan=plan, **HP))
    f64 = dict(out_dtype="float32", acc=np.float64)
    y_ref, dA_ref = oracle.gmm(x, A, gs, **f64), oracle.tgmm(x, dy, gs, **f64)
    # 16-bit results: one rounding to a significand of 8 or 11 bits (at most 2^-8 or 2^-11 of the value) on top of fp32 sums
    # of at most 577 products (577 x 2^-24 = 3.5e-5); float32 results: the sums alone
    eps = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -11, "float32": 0.0}[rounding] if storage != torch.float32 else 0.0
    eps += 577 * 2.0 ** -24
    for name, got in (("y", y), ("y (trans_rhs)", yt)):
        assert np.all(np.isnan(got[hit])), f"{name}: the poisoned group's rows"
        live = clean & (np.arange(m) < total)
        err = np.linalg.norm(got[live] - y_ref[live], axis=1) / np.linalg.norm(y_ref[live], axis=1)
        assert err.max() < eps, f"{name}: {err.max()} >= {eps}"
        assert not np.any(got[total:]), f"{name}: tail rows"
    for i in range(g):
        if i == poisoned:
            continue
        if gs[i] == 0:
            assert not np.any(dA[i])
        else:
            err = np.linalg.norm(dA[i] - dA_ref[i]) / np.linalg.norm(dA_ref[i])
            assert err < eps, f"dA[{i}]: {err} >= {eps}"


@pytest.mark.parametrize("vid,vname,dtype", [v for v in VARIANTS if "256x256" in v[1] or "128x128" in v[1]],
                         ids=[v[1] for v in VARIANTS if "256x256" in v[1] or "128x128" in v[1]])
@pytest.mark.parametrize("trans_rhs", [False, True])
def test_row_tiles_shorter_than_the_tile(vid, vname, dtype, trans_rhs):
    """A gmm launch computes a row tile of few rows at a multiple of 64: every height and one row to either side of it, as a
    group's only tile and behind a whole one; the rows behind a group belong to the next and must stay its own."""
    print(f"short row tiles, variant {vname} trans_rhs {trans_rhs}", flush=True)
    rounding, storage, compute = KINDS[dtype]
    gs = np.array([1, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 256 + 1, 256 + 64, 256 + 65, 0, 2 * 256 + 130], np.int32)
    g, m, k, n = len(gs), int(gs.sum()) + 3, 200, 264
    rng = np.random.default_rng(vid)
    r = lambda a: oracle.round_to(a, rounding)
    x, A = r(rng.normal(size=(m, k))), r(rng.normal(size=(g, k, n)) / np.sqrt(k))
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().to(storage)
    y = util.to_np(ops._gmm_fwd(dev(x), dev(np.swapaxes(A, 1, 2) if trans_rhs else A), torch.from_numpy(gs).cuda(), trans_rhs=trans_rhs,
                                compute_dtype=compute, plan=_capi.Plan(vid), **HP))
    ref = oracle.gmm(x, A, gs, out_dtype="float32", acc=np.float64)
    # the bound of the test above, for 200 products
    eps = {"bfloat16": 2.0 ** -8, "float16": 2.0 ** -11, "float32": 0.0}[rounding] if storage != torch.float32 else 0.0
    eps += 200 * 2.0 ** -24
    err = np.linalg.norm(y[:m - 3] - ref[:m - 3], axis=1) / np.linalg.norm(ref[:m - 3], axis=1)
    assert err.max() < eps, f"{err.max()} >= {eps} in row {err.argmax()}"
    assert not np.any(y[m - 3:])


@pytest.mark.parametrize("vid,vname", [v[:2] for v in VARIANTS if v[1].startswith("fr")], ids=[v[1] for v in VARIANTS if v[1].startswith("fr")])
@pytest.mark.parametrize("k,trans_rhs", [(799, False), (800, True), (800, False), (1025, True), (2111, False), (4096, True)])
def test_float32_last_round_cut_along_k(vid, vname, k, trans_rhs):
    """float32 tiles left over from whole rounds are computed in pieces of the contraction from k = 800 on: odd k and n,
    groups of one row and of a tile's, against the oracle and against the uncut launch; the same bits on a second call."""
    print(f"float32 k-split, variant {vname} k {k} trans_rhs {trans_rhs}", flush=True)
    gs = np.array([1, 0, 130, 257, 64, 3], np.int32)
    g, m, n = len(gs), int(gs.sum()) + 5, 201
    rng = np.random.default_rng(k)
    x, A = rng.normal(size=(m, k)).astype(np.float32), (rng.normal(size=(g, k, n)) / np.sqrt(k)).astype(np.float32)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    args = (dev(x), dev(np.swapaxes(A, 1, 2) if trans_rhs else A), dev(gs))
    run = lambda split: ops._gmm_fwd(*args, trans_rhs=trans_rhs, compute_dtype=None, plan=_capi.Plan(vid, split_k=split), **HP)
    cut, again, whole = run(0), run(0), run(-1)
    assert torch.equal(cut, again)
    assert torch.equal(cut, whole) == (k < 800)
    ref = oracle.gmm(x, A, gs, out_dtype="float32", acc=np.float64)
    total = int(gs.sum())
    for y in (util.to_np(cut), util.to_np(whole)):
        err = np.linalg.norm(y[:total] - ref[:total], axis=1) / np.linalg.norm(ref[:total], axis=1)
        assert err.max() < k * 2.0 ** -24, f"{err.max()} in row {err.argmax()}"  # k float32 additions
        assert not np.any(y[total:])


@pytest.mark.parametrize("k,n", [(5, 16), (16, 3), (7, 100), (1, 1)])
@pytest.mark.parametrize("blocks", [(128, 64, 128), (256, 256, 256)])
@pytest.mark.parametrize("trans_rhs", [False, True])
def test_explicit_blocks_on_rows_of_a_few_elements(k, n, blocks, trans_rhs):
    """Explicit block sizes ask for a large tile; rows of fewer than 8 elements get the one that takes them, forward and in
    both gradients."""
    print(f"explicit blocks {blocks} k {k} n {n} trans_rhs {trans_rhs}", flush=True)
    gs = np.array([20, 0, 37, 3], np.int32)
    g, m = len(gs), int(gs.sum()) + 4
    rng = np.random.default_rng(k * 100 + n)
    r = lambda a: oracle.round_to(a, "bfloat16")
    x, A, dy = r(rng.normal(size=(m, k))), r(rng.normal(size=(g, k, n))), r(rng.normal(size=(m, n)))
    block_m, block_k, block_n = blocks
    xt = util.bf16_dev(x).requires_grad_()
    At = util.bf16_dev(np.ascontiguousarray(np.swapaxes(A, 1, 2)) if trans_rhs else A).requires_grad_()
    y = rd.gmm(xt, At, torch.from_numpy(gs).cuda(), block_m=block_m, block_k=block_k, block_n=block_n, trans_rhs=trans_rhs)
    dx, dA = torch.autograd.grad(y, (xt, At), util.bf16_dev(dy))
    f64 = dict(out_dtype="float32", acc=np.float64)
    dA = dA.transpose(1, 2) if trans_rhs else dA
    for name, got, ref in (("y", y.detach(), oracle.gmm(x, A, gs, **f64)), ("dx", dx, oracle.gmm(dy, np.swapaxes(A, 1, 2), gs, **f64)),
                           ("dA", dA, oracle.tgmm(x, dy, gs, **f64))):
        # one rounding to a significand of 8 bits on top of float32 sums
        assert np.linalg.norm(util.to_np(got) - ref) <= 2.0 ** -8 * np.linalg.norm(ref), name
