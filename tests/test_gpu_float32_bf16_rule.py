"""float32 multiplied in bfloat16 (compute_dtype): sizes that the default rule gives to each of its tiles, at 16-byte pitches and at odd ones."""

import numpy as np
import pytest
import torch

import gpu_ragged_dot_amd as rd
from gpu_ragged_dot_amd import _capi
from oracle import ragged_dot_oracle as oracle
from tests import util

# m, k, n, g, tile of gmm, tile of tgmm: two rounds and four of 256 x 256 tiles of tgmm, few rows, few columns, short contractions
SIZES = [(9000, 1000, 1504, 6, "cr256x256x32_w2x4", "cr128x128x32_w2x2"), (6000, 1000, 1504, 40, "cr256x256x32_w2x4", "cr256x256x32_w2x4"),
         (1270, 1000, 1504, 40, "cr128x128x32_w2x2", "cr128x128x32_w2x2"), (255, 520, 496, 32, "cr128x128x32_w2x2", "c64x64x32_w2x2"),
         (1500, 512, 48, 4, "c64x64x32_w2x2", "cr128x128x32_w2x2"), (240, 512, 64, 4, "cr128x128x32_w2x2", "c64x64x32_w2x2"),
         (9000, 1001, 1515, 6, "cs256x256x32_w2x4", "cs128x128x32_w2x2"), (2800, 265, 703, 45, "cs128x128x32_w2x2", "c64x64x32_w2x2"),
         (300, 31, 99, 2, "c64x64x32_w2x2", "c64x64x32_w2x2"), (300, 33, 99, 2, "c64x64x32_w2x2", "c64x64x32_w2x2"),
         (300, 7, 99, 2, "c64x64x32_w2x2", "c64x64x32_w2x2"),
         # brief launches, and their neighbours with a few more tiles, a longer contraction or longer groups
         (1000, 120, 960, 4, "cr128x128x32_w2x2", "cr128x128x32_w2x2"), (1000, 120, 896, 4, "c64x64x32_w2x2", "cr128x128x32_w2x2"),
         (1000, 136, 896, 4, "cr128x128x32_w2x2", "cr128x128x32_w2x2"), (768, 512, 512, 6, "cr128x128x32_w2x2", "c64x64x32_w2x2"),
         (768, 576, 512, 7, "cr128x128x32_w2x2", "c64x64x32_w2x2"), (768, 576, 576, 7, "cr128x128x32_w2x2", "cr128x128x32_w2x2"),
         (900, 250, 900, 2, "c64x64x32_w2x2", "cs128x128x32_w2x2"), (900, 250, 1100, 2, "cs128x128x32_w2x2", "cs128x128x32_w2x2"),
         (900, 270, 900, 2, "cs128x128x32_w2x2", "cs128x128x32_w2x2"), (900, 509, 900, 8, "cs128x128x32_w2x2", "c64x64x32_w2x2"),
         (900, 509, 1100, 8, "cs128x128x32_w2x2", "cs128x128x32_w2x2"), (9000, 45, 1900, 5, "c64x64x32_w2x2", "cs128x128x32_w2x2"),
         (9000, 45, 1700, 5, "cs128x128x32_w2x2", "cs128x128x32_w2x2"), (760, 509, 900, 5, "cs128x128x32_w2x2", "cs128x128x32_w2x2"),
         (760, 450, 700, 5, "cs128x128x32_w2x2", "c64x64x32_w2x2"), (760, 125, 700, 3, "c64x64x32_w2x2", "c64x64x32_w2x2")]
OPS = (_capi.OP_GMM, _capi.OP_TGMM)


@pytest.mark.parametrize("m,k,n,g,gmm,tgmm", SIZES)
def test_default_rule(m, k, n, g, gmm, tgmm):
    names = [_capi.variants()[_capi.default_plan(op, m, k, n, g, _capi.RD_DTYPE_F32_BF16).variant].name.decode() for op in OPS]
    assert names == [gmm, tgmm]


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,g,gmm,tgmm", SIZES)
def test_products_of_the_default_tiles(m, k, n, g, gmm, tgmm):
    rng = np.random.default_rng(m + k)
    p = np.exp(rng.standard_normal(g))
    gs = rng.multinomial(m - 9, p / p.sum()).astype(np.int32)
    if g > 2:
        gs[1] = 0
    live = int(gs.sum())
    r = lambda a: oracle.round_to(a.astype(np.float32), "bfloat16")
    x, A, dy = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((g, k, n)).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    xd, Ad, dyd, gsd = dev(x), dev(A), dev(dy), torch.from_numpy(gs).cuda()
    bf16 = dict(compute_dtype=torch.bfloat16)
    # float32 sums of the rounded operands: a rounding of the running sum for every product
    wide = dict(out_dtype="float32", acc=np.float64)
    y_ref, dA_ref = oracle.gmm(r(x), r(A), gs, **wide), oracle.tgmm(r(x), r(dy), gs, **wide)
    for y in (rd.ragged_dot(xd, Ad, gsd, **bf16), rd.ragged_dot(xd, Ad.mT.contiguous(), gsd, trans_rhs=True, **bf16)):
        y = util.to_np(y)
        err = np.linalg.norm(y[:live] - y_ref[:live], axis=1) / np.linalg.norm(y_ref[:live], axis=1)
        assert err.max() < (k + 1) * 2.0 ** -24 and not np.any(y[live:])
    dA = util.to_np(rd.tgmm(xd, dyd, gsd, **bf16))
    some = gs > 0
    err = np.linalg.norm((dA - dA_ref)[some], axis=(1, 2)) / np.linalg.norm(dA_ref[some], axis=(1, 2))
    assert np.all(err < (gs[some] + 1) * 2.0 ** -24) and not np.any(dA[~some])
