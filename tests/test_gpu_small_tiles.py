"""The core of rd_gemm_ws.h (128- and 64-row tiles for launches that do not fill the device) against the oracle.

Sizes where they can go wrong: contractions of less than one slab, around one slab and around the ring's depth (where the
unconditional loop takes over), tile edges, groups of 0, 1 and one more than a tile's rows.  One group's operands are NaN: nothing of it may reach the others.
"""

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi, ops
from oracle import ragged_dot_oracle as oracle
from tests import util

gpu = pytest.mark.gpu

HP = dict(block_m=64, block_k=64, block_n=64, interpret=False, acc_dtype=torch.float32, chunk_m=512)
VARIANTS = [(v.id, v.name.decode(), v.dtype, v.tile_m) for v in _capi.variants() if v.name.decode().startswith(("v", "hv"))]
KINDS = {_capi.RD_DTYPE_BF16: ("bfloat16", torch.bfloat16, 2.0 ** -8), _capi.RD_DTYPE_F16: ("float16", torch.float16, 2.0 ** -11)}
# (k, n): slabs of 32 or 64, rings of 3, 5 and 6
SHAPES = [(8, 8), (32, 120), (40, 136), (64, 256), (72, 264), (96, 128), (136, 520), (184, 8), (256, 72), (320, 136), (328, 264),
          (384, 128), (456, 200), (520, 264)]


def _dev(a, storage):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().to(storage)


@gpu
@pytest.mark.parametrize("vid,vname,dtype,tile_m", VARIANTS, ids=[v[1] for v in VARIANTS])
@pytest.mark.parametrize("k,n", SHAPES, ids=[f"k{k}n{n}" for k, n in SHAPES])
def test_small_tile_edges(vid, vname, dtype, tile_m, k, n):
    print(f"variant {vname} k {k} n {n}", flush=True)
    rounding, storage, eps = KINDS[dtype]
    gs = np.array([257, 0, 1, 63, 40, 129, 7, 393], np.int32)  # tgmm's contractions too: 393 is 12 slabs of 32 and 9 rows
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
    gs_t, plan = torch.from_numpy(gs).cuda(), _capi.Plan(vid)
    y = util.to_np(ops._gmm_fwd(_dev(x_in, storage), _dev(A_in, storage), gs_t, trans_rhs=False, compute_dtype=None, plan=plan, **HP))
    yt = util.to_np(ops._gmm_fwd(_dev(x_in, storage), _dev(np.swapaxes(A_in, 1, 2), storage), gs_t, trans_rhs=True, compute_dtype=None,
                                 plan=plan, **HP))
    f64 = dict(out_dtype="float32", acc=np.float64)
    y_ref, dA_ref = oracle.gmm(x, A, gs, **f64), oracle.tgmm(x, dy, gs, **f64)
    # one rounding to a significand of 8 or 11 bits on top of fp32 sums of at most 520 products
    bound = eps + 520 * 2.0 ** -24
    for name, got in (("y", y), ("y (trans_rhs)", yt)):
        assert np.all(np.isnan(got[hit])), f"{name}: the poisoned group's rows"
        live = clean & (np.arange(m) < total)
        err = np.linalg.norm(got[live] - y_ref[live], axis=1) / np.linalg.norm(y_ref[live], axis=1)
        assert err.max() < bound, f"{name}: {err.max()} >= {bound}"
        assert not np.any(got[total:]), f"{name}: tail rows"
    dA = util.to_np(ops._tgmm_fwd(_dev(x_in, storage), _dev(dy_in, storage), gs_t, compute_dtype=None, plan=plan, **HP))
    for i in range(g):
        if i == poisoned:
            continue
        if gs[i] == 0:
            assert not np.any(dA[i])
        else:
            err = np.linalg.norm(dA[i] - dA_ref[i]) / np.linalg.norm(dA_ref[i])
            assert err < bound, f"dA[{i}]: {err} >= {bound}"


def test_default_plans_name_a_tile_that_takes_the_product():
    """Every branch of the default rules, over sizes from one row or column up: the variant named takes the call."""
    rng = np.random.default_rng(5)
    seen = set()
    for _ in range(6000):
        op, g = int(rng.integers(0, 3)), int(np.exp(rng.uniform(0, np.log(300))))
        m, k, n = (int(np.exp(rng.uniform(0, np.log(top)))) for top in (40000, 17000, 17000))
        if rng.random() < 0.8:
            k, n = (k + 7) // 8 * 8, (n + 7) // 8 * 8
        for dtype in (_capi.RD_DTYPE_BF16, _capi.RD_DTYPE_F16):
            plan = _capi.default_plan(op, m, k, n, g, dtype)
            assert _capi.lib.rd_variant_takes(plan.variant, op, m, k, n, dtype) == _capi.RD_OK, (op, m, k, n, g, dtype)
            seen.add(_capi.variants()[plan.variant].name.decode())
    missing = {v[1] for v in VARIANTS} - seen
    assert not missing, missing


def test_default_tiles_by_rounds():
    """Which core the rules name where a launch is two thirds to one round of 256 x 256 tiles, a round and a bit, or several rounds; and
    for groups of a quarter to half a tile's height whose weights the last-level cache holds."""
    name = lambda op, m, k, n, g: _capi.variants()[_capi.default_plan(op, m, k, n, g, _capi.RD_DTYPE_BF16).variant].name.decode()
    assert name(1, 4096, 4096, 2048, 16) == "w256x256x32_w2x2_s5"      # 192 expected tiles
    assert name(1, 5120, 4096, 2560, 20) == "v128x256x64_w2x2_s3"      # 300
    assert name(1, 5476, 10296, 3256, 39) == "w256x256x32_w2x2_s5"     # 540
    assert name(1, 2560, 1024, 2048, 32) == "q256x256x32_w2x4"         # 80 rows a group, 134 MB of weights
    assert name(0, 2560, 1024, 2048, 32) == "q256x256x32_w2x4"
    assert name(1, 2560, 4096, 4096, 32) == "w256x256x32_w2x2_s5"      # 80 rows, 1.1 GB
    assert name(1, 2560, 1024, 4096, 64) == name(0, 2560, 1024, 4096, 64) == "w256x256x32_w2x2_s5"  # 40 rows
    assert name(2, 32768, 768, 2048, 128) == "v128x256x32_w2x2_s3"     # tgmm, x of 50 MB
    assert name(2, 32768, 2048, 768, 128) == "p256x256x32_w2x4_s4"     # 134 MB
