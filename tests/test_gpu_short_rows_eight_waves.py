"""Row tiles of at most 128 rows on the eight-wave core with a ring per operand run on routines of 64 or 128 rows: group sizes on
both sides of each limit, a group's only tile and its last one, contractions around the slab and the rings' depth, cut along K and
not, against the oracle."""

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi, ops
from oracle import ragged_dot_oracle as oracle
from tests import util

gpu = pytest.mark.gpu

HP = dict(block_m=64, block_k=64, block_n=64, interpret=False, acc_dtype=torch.float32, chunk_m=512)
VID = next(v.id for v in _capi.variants() if v.name.decode() == "q256x256x32_w2x4")


@gpu
@pytest.mark.parametrize("trans_rhs", [False, True], ids=["nn", "nt"])
@pytest.mark.parametrize("k,split_k", [(8, 0), (64, 0), (72, 0), (136, 0), (192, 0), (264, 0), (520, 0), (1096, 2), (2056, 3)])
def test_short_row_tiles(k, split_k, trans_rhs):
    print(f"k {k} split_k {split_k} trans_rhs {trans_rhs}", flush=True)
    gs = np.array([1, 64, 65, 0, 128, 129, 257, 320, 321, 384, 385, 33], np.int32)
    n, g, total, poisoned, tail = 264, len(gs), int(gs.sum()), 7, 5
    m = total + tail
    rng = np.random.default_rng(k)
    r = lambda a: oracle.round_to(a, "bfloat16")
    x, A = r(rng.normal(size=(m, k))), r(rng.normal(size=(g, k, n)) / np.sqrt(k))
    first = int(gs[:poisoned].sum())
    x_in, A_in = x.copy(), A.copy()
    x_in[first:first + gs[poisoned]], A_in[poisoned] = np.nan, np.nan
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().to(torch.bfloat16)
    w = np.swapaxes(A_in, 1, 2) if trans_rhs else A_in
    y = util.to_np(ops._gmm_fwd(dev(x_in), dev(w), torch.from_numpy(gs).cuda(), trans_rhs=trans_rhs, compute_dtype=None,
                                plan=_capi.Plan(VID, split_k=split_k), **HP))
    ref = oracle.gmm(x, A, gs, out_dtype="float32", acc=np.float64)
    live = np.arange(m) < total
    live[first:first + gs[poisoned]] = False
    assert np.all(np.isnan(y[first:first + gs[poisoned]])) and not np.any(y[total:])
    err = np.linalg.norm(y[live] - ref[live], axis=1) / np.linalg.norm(ref[live], axis=1)
    assert err.max() < 2.0 ** -8 + k * 2.0 ** -24, err.max()  # one rounding of the result on top of fp32 sums of k products


def test_one_row_tile_per_band():
    """The walk of many groups of about one row tile, at the edges of its range."""
    walk = lambda m, g: (lambda p: (_capi.variants()[p.variant].name.decode(), p.group_m, p.group_n))(
        _capi.default_plan(0, m, 3072, 1024, g, _capi.RD_DTYPE_BF16))
    assert walk(24576, 96) == ("q256x256x32_w2x4", 1, 8)
    assert walk(192 * 96, 96)[1:] == (1, 8) and walk(384 * 96, 96)[1:] == (1, 8)
    assert walk(192 * 96 - 1, 96)[1] != 1 and walk(384 * 96 + 1, 96)[1] != 1 and walk(256 * 63, 63)[1] != 1
