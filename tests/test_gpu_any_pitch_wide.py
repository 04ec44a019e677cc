"""The 128 x 256 tile of the any-pitch core: sizes that the default rules give to it, and their neighbours on either side of the rule's lines."""

import numpy as np
import pytest
import torch

import gpu_ragged_dot_amd as rd
from gpu_ragged_dot_amd import _capi
from oracle import ragged_dot_oracle as oracle
from tests import util

pytestmark = pytest.mark.gpu

# m, k, n, g, taken: a round of tiles, two rounds; contractions and tile counts below the lines; short groups
SIZES = [(2178, 831, 2203, 3, True), (3000, 701, 1601, 4, True), (3900, 1501, 1030, 5, True), (6700, 303, 1799, 3, True),
         (2178, 699, 2203, 3, False), (1100, 831, 2203, 3, False), (2178, 831, 2203, 30, False),
         (3000, 701, 1301, 4, True), (2800, 1001, 1301, 4, False)]  # 156 and 144 tiles


# m, k, n, g, tile: few tiles and contractions on either side of the 64 x 64 tile's lines; up to four rounds of 128 x 256 tiles, and more
FEW = [(300, 2049, 301, 3, "r128x128x64_w2x2"), (300, 1025, 301, 3, "64x64x32_w2x2"), (1000, 1025, 501, 3, "r128x128x64_w2x2"),
       (1000, 513, 501, 3, "64x64x32_w2x2"), (2100, 513, 501, 3, "r128x128x64_w2x2"), (9001, 777, 1999, 12, "r128x256x64_w2x4"),
       (9001, 777, 3999, 12, "r256x256x64_w2x2")]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("m,k,n,g,taken", SIZES)
def test_default_rule(m, k, n, g, taken, dtype):
    _check(m, k, n, g, dtype, lambda name: name.endswith("r128x256x64_w2x4") == taken)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("m,k,n,g,tile", FEW)
def test_few_tiles(m, k, n, g, tile, dtype):
    _check(m, k, n, g, dtype, lambda name: name.endswith(tile))


def _check(m, k, n, g, dtype, expected):
    rng = np.random.default_rng(m + k)
    p = np.exp(rng.standard_normal(g))
    gs = rng.multinomial(m - 9, p / p.sum()).astype(np.int32)
    code = _capi.RD_DTYPE_BF16 if dtype == torch.bfloat16 else _capi.RD_DTYPE_F16
    names = [v.name.decode() for v in _capi.variants()]
    for op in (_capi.OP_GMM, _capi.OP_GMM_TRANS):
        name = names[_capi.default_plan(op, m, k, n, g, code).variant]
        assert expected(name), name
    rounding = "bfloat16" if dtype == torch.bfloat16 else "float16"
    x = oracle.round_to(rng.standard_normal((m, k)).astype(np.float32), rounding)
    A = oracle.round_to((rng.standard_normal((g, k, n)) / np.sqrt(k)).astype(np.float32), rounding)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().to(dtype)
    xd, Ad, gsd = dev(x), dev(A), torch.from_numpy(gs).cuda()
    ref = oracle.gmm(x, A, gs, out_dtype="float32", acc=np.float64)
    live = int(gs.sum())
    # one rounding to 8 or 11 bits, and float32 sums of k products
    eps = (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) + k * 2.0 ** -24
    for y in (rd.ragged_dot(xd, Ad, gsd), rd.ragged_dot(xd, Ad.mT.contiguous(), gsd, trans_rhs=True)):
        y = util.to_np(y)
        err = np.linalg.norm(y[:live] - ref[:live], axis=1) / np.linalg.norm(ref[:live], axis=1)
        assert err.max() < eps and not np.any(y[live:])


# m, k, n, g, whether tgmm takes the 128 x 128 tile: rows of a group times tiles, rows alone, few columns
@pytest.mark.parametrize("m,k,n,g,taken", [(9000, 65, 99, 3, False), (9000, 165, 199, 3, True), (9000, 301, 77, 3, True), (4000, 301, 77, 16, False),
                                           (9000, 301, 55, 8, False), (1304, 137, 1358, 4, False), (3000, 301, 301, 5, False),
                                           (3000, 601, 601, 5, True), (3000, 401, 501, 3, False), (3000, 701, 901, 3, True)])
def test_tgmm_few_tiles(m, k, n, g, taken):
    name = _capi.variants()[_capi.default_plan(_capi.OP_TGMM, m, k, n, g, _capi.RD_DTYPE_BF16).variant].name.decode()
    assert name == ("r128x128x64_w2x2" if taken else "s64x64x32_w2x2")
    rng = np.random.default_rng(m + k)
    gs = rng.multinomial(m - 9, np.ones(g) / g).astype(np.int32)
    x, dy = (oracle.round_to(rng.standard_normal(s).astype(np.float32), "bfloat16") for s in ((m, k), (m, n)))
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(torch.bfloat16)
    dA = util.to_np(rd.tgmm(dev(x), dev(dy), torch.from_numpy(gs).cuda()))
    ref = oracle.tgmm(x, dy, gs, out_dtype="float32", acc=np.float64)
    err = np.linalg.norm(dA - ref, axis=(1, 2)) / np.linalg.norm(ref, axis=(1, 2))
    assert err.max() < 2.0 ** -8 + gs.max() * 2.0 ** -24  # one rounding to 8 bits, and float32 sums
