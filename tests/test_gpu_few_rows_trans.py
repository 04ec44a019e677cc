"""trans_rhs over groups of a few rows: the tile that the default rule takes on either side of its lines (rows of a group, the weights' pitch).  Operands of -1, 0
and 1 and outputs below 256, so that the products have to come out exactly."""

import numpy as np
import pytest
import torch

import gpu_ragged_dot_amd as rd
from gpu_ragged_dot_amd import _capi
from oracle import ragged_dot_oracle as oracle
from tests import util

# m, k, n, g, the 64 x 64 tile of the core for unfilled launches or the four-wave core
SIZES = [(1500, 1000, 768, 100, True), (1590, 3064, 776, 100, True), (1601, 1000, 776, 100, False), (1500, 2048, 768, 100, False)]


@pytest.mark.parametrize("dtype,prefix", [(_capi.RD_DTYPE_BF16, ""), (_capi.RD_DTYPE_F16, "h")])
@pytest.mark.parametrize("m,k,n,g,small", SIZES)
def test_default_rule(m, k, n, g, small, dtype, prefix):
    plan = _capi.default_plan(_capi.OP_GMM_TRANS, m, k, n, g, dtype)
    assert plan.decode_nb == 0
    assert _capi.variants()[plan.variant].name.decode() == prefix + ("v64x64x64_w2x2_s5" if small else "w256x256x32_w2x2_s5")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("m,k,n,g,small", SIZES)
def test_whole_numbers_come_out_exactly(m, k, n, g, small, dtype):
    rng = np.random.default_rng(m + k)
    gs = rng.multinomial(m - 9, np.ones(g) / g).astype(np.int32)
    gs[3], gs[4] = 0, gs[3] + gs[4]
    x = rng.integers(-1, 2, size=(m, k)).astype(np.float32)
    x[:, 200:] = 0  # sums of at most 200
    A = rng.integers(-1, 2, size=(g, n, k)).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).cuda().to(dtype)
    y = rd.ragged_dot(dev(x), dev(A), torch.from_numpy(gs).cuda(), trans_rhs=True)
    assert np.array_equal(util.to_np(y), oracle.gmm(x, A, gs, trans_rhs=True, out_dtype="float32"))
