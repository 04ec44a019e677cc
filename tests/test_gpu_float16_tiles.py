"""The float16 tiles that follow the bfloat16 ones: row tiles of every height class, partial column tiles, short contractions, the last round cut
along K.  Operands of -1, 0 and 1, so that every sum is a whole number below 2048 and has to come out exactly."""

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi, ops
from oracle import ragged_dot_oracle as oracle
from tests import util

NAMES = ["hp256x256x32_w2x4_s4", "hq256x256x32_w2x4", "hp128x256x32_w2x4_s3", "hd128x128x32_w2x2_s3", "ht64x64x64_w2x2"]
ROWS = [0, 1, 31, 64, 65, 128, 129, 255, 0, 256, 257, 513, 7]
HP = dict(block_m=64, block_k=64, block_n=64, interpret=False, compute_dtype=None, acc_dtype=torch.float32, chunk_m=512)


def _signs(rng, shape):
    return rng.integers(-1, 2, size=shape).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("k,n", [(8, 264), (40, 64), (264, 136), (1032, 520)])
@pytest.mark.parametrize("name", NAMES)
def test_whole_numbers_come_out_exactly(name, k, n):
    rng = np.random.default_rng(k + n)
    gs = np.array(ROWS, np.int32)
    live = int(gs.sum())
    m, g = live + 30, len(ROWS)
    x, A, dy = _signs(rng, (m, k)), _signs(rng, (g, k, n)), _signs(rng, (m, n))
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(torch.float16)
    vid = next(v.id for v in _capi.variants() if v.name.decode() == name)
    xd, gsd, dyd = dev(x), torch.from_numpy(gs).cuda(), dev(dy)
    y_ref = oracle.gmm(x, A, gs, out_dtype="float32")
    for trans_rhs in (False, True):
        w = dev(np.swapaxes(A, 1, 2) if trans_rhs else A)
        for split_k in (-1, 0, 2):
            y = ops._gmm_fwd(xd, w, gsd, **HP, trans_rhs=trans_rhs, plan=_capi.Plan(vid, 0, 0, 0, split_k))
            assert y.dtype == torch.float16 and np.array_equal(util.to_np(y), y_ref), (trans_rhs, split_k)
    dA = ops._tgmm_fwd(xd, dyd, gsd, **HP, plan=_capi.Plan(vid))
    assert np.array_equal(util.to_np(dA), oracle.tgmm(x, dy, gs, out_dtype="float32"))


# op, m, k, n, g, tile: either side of the rule's lines
RULE = [(_capi.OP_TGMM, 8192, 7168, 2048, 32, "hp256x256x32_w2x4_s4"), (_capi.OP_TGMM, 32768, 7168, 2048, 32, "hw256x256x32_w2x2_s5"),
        (_capi.OP_TGMM, 1291, 832, 2240, 75, "hd128x128x32_w2x2_s3"), (_capi.OP_TGMM, 2619, 448, 304, 37, "hv128x128x32_w2x2_s5"),
        (_capi.OP_TGMM, 1497, 272, 480, 4, "ht64x64x64_w2x2"), (_capi.OP_GMM_TRANS, 24460, 784, 1376, 85, "hq256x256x32_w2x4"),
        (_capi.OP_GMM, 6849, 2512, 10736, 27, "hq256x256x32_w2x4"), (_capi.OP_GMM, 23150, 1520, 5504, 11, "hw256x256x32_w2x2_s5")]


@pytest.mark.parametrize("op,m,k,n,g,name", RULE)
def test_default_rule(op, m, k, n, g, name):
    assert _capi.variants()[_capi.default_plan(op, m, k, n, g, _capi.RD_DTYPE_F16).variant].name.decode() == name
