"""float8: sizes that the default rule gives to each of the direct-to-LDS tiles.  Operands of -1, 0 and 1 and short contractions, so that every sum is a
whole number that bfloat16 holds."""

import numpy as np
import pytest
import torch

import gpu_ragged_dot_amd as rd
from gpu_ragged_dot_amd import _capi
from oracle import ragged_dot_oracle as oracle
from tests import util

TILES = {256: "x256x256x64_w2x4_s4", 128: "x128x256x64_w2x4_s3", 64: "x64x256x64_w1x4_s8"}
# m, k, n, g, tile of gmm, tile of gmm on weights [g, n, k]
SIZES = [(2283, 240, 3152, 7, 128, 128), (9000, 208, 4096, 5, 128, 128), (300, 256, 528, 2, 64, 64), (16384, 4096, 14336, 8, 256, 256),
         (2283, 1680, 3152, 7, 256, 256), (596, 6400, 288, 213, 128, 128),
         (1000, 208, 3840, 2, 64, 64), (1000, 208, 4096, 2, 128, 128), (64, 16, 64, 3, 64, 64)]  # up to a round of 64 x 256 tiles


@pytest.mark.parametrize("m,k,n,g,gmm,gmm_t", SIZES)
def test_default_rule(m, k, n, g, gmm, gmm_t):
    for op, tile in ((_capi.OP_GMM, gmm), (_capi.OP_GMM_TRANS, gmm_t)):
        assert _capi.variants()[_capi.default_plan(op, m, k, n, g, _capi.RD_DTYPE_F8E4M3_BF16).variant].name.decode() == TILES[tile]


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,n,g,gmm,gmm_t", [c for c in SIZES if c[1] <= 256])
def test_whole_numbers_come_out_exactly(m, k, n, g, gmm, gmm_t):
    rng = np.random.default_rng(m + k)
    p = np.exp(rng.standard_normal(g))
    gs = rng.multinomial(m - 9, p / p.sum()).astype(np.int32)
    x, A = (rng.integers(-1, 2, size=s).astype(np.float32) for s in ((m, k), (g, k, n)))  # sums of at most 240: 8 bits
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(torch.float8_e4m3fn)
    ref = oracle.gmm(x, A, gs, out_dtype="float32")
    gsd = torch.from_numpy(gs).cuda()
    assert np.array_equal(util.to_np(rd.ragged_dot(dev(x), dev(A), gsd)), ref)
    assert np.array_equal(util.to_np(rd.ragged_dot(dev(x), dev(np.swapaxes(A, 1, 2)), gsd, trans_rhs=True)), ref)
