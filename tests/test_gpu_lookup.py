"""Products whose work-groups look their tile up in group_sizes themselves (no map kernel) against the same launch with the
map built (a plan that forbids the K-split keeps it): same tiles, same bits.  Group counts on both sides of what one wave
load, and all of them, cover; empty groups first, last and in runs; a zero tail; all groups empty."""

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi, ops
from oracle import ragged_dot_oracle as oracle
from tests import util

pytestmark = pytest.mark.gpu

HP = dict(block_m=64, block_k=64, block_n=64, interpret=False, compute_dtype=None, acc_dtype=torch.float32, chunk_m=512)


@pytest.mark.parametrize("g", [1, 63, 64, 65, 129, 255, 256, 257, 300])
@pytest.mark.parametrize("fill", ["some", "none"])
def test_lookup_matches_the_map(g, fill):
    print(f"lookup g {g} fill {fill}", flush=True)
    rng = np.random.default_rng(g)
    gs = rng.integers(0, 40, size=g).astype(np.int32) * (rng.random(g) < 0.6)
    gs[rng.integers(0, g)] = 200
    if g > 3:
        gs[0], gs[-1] = 0, 0
    if fill == "none":
        gs[:] = 0
    gs = gs.astype(np.int32)
    total = int(gs.sum())
    m, k, n = total + 70, 72, 136
    lhs, rhs, dout = (oracle.round_to(rng.normal(size=s).astype(np.float32), "bfloat16") for s in ((m, k), (g, k, n), (m, n)))
    x, A, d, gs_t = util.bf16_dev(lhs), util.bf16_dev(rhs), util.bf16_dev(dout), torch.from_numpy(gs).cuda()
    for name in ("t64x64x64_w2x2", "t32x256x64_w1x4", "s64x64x32_w2x2", "d128x128x32_w2x2_s3"):
        vid = [v.id for v in _capi.variants() if v.name.decode() == name][0]
        y, y_map = (ops._gmm_fwd(x, A, gs_t, trans_rhs=False, plan=_capi.Plan(vid, 3, 0, 2, split_k=s), **HP) for s in (0, -1))
        assert torch.equal(y, y_map), name
        util.assert_close_rows(util.to_np(y), oracle.gmm(lhs, rhs, gs), total, util.BF16_EPS, name) if total else None
        assert not torch.any(y[total:]), name
        dA, dA_map = (ops._tgmm_fwd(x, d, gs_t, plan=_capi.Plan(vid, 4, 0, order), **HP) for order in (-1, 1))
        assert torch.equal(dA, dA_map), name
        assert not torch.any(dA[gs_t == 0]), name
