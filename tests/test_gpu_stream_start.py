"""The streaming tiles of trans_rhs begin at slabs of their own (gemm_tile_dlds()) where the contraction is a multiple of
kRotatePitch = 2048: whole contractions, which then have 32 slabs and more, and pieces of one that is cut along K, whose counts
of slabs are odd ones too, against the oracle.  (Starts in contractions of fewer slabs than the ring holds, and last slabs that
are not full, which no such contraction has: the loaders' host check.)  Other contractions run on the same routines from their
first slab: one slab, around the ring's depth, a last slab that is not full."""

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi, ops
from oracle import ragged_dot_oracle as oracle
from tests import util

pytestmark = pytest.mark.gpu

HP = dict(block_m=64, block_k=64, block_n=64, interpret=False, acc_dtype=torch.float32, chunk_m=512)
CORES = [("w256x256x32_w2x2_s5", "bfloat16", torch.bfloat16, 2.0 ** -8), ("hw256x256x32_w2x2_s5", "float16", torch.float16, 2.0 ** -11)]


def _vid(name):
    return next(v.id for v in _capi.variants() if v.name.decode() == name)


def _dev(a, storage):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().to(storage)


# (k, split_k), slabs of 64: 2048 in pieces of 10, 11 and 11, 4096 of 21, 21 and 22, 6144 of 24; 8192 is cut by default
@pytest.mark.parametrize("name,rounding,storage,eps", CORES)
@pytest.mark.parametrize("k,split_k", [(2048, -1), (4096, -1), (6144, -1), (2048, 3), (4096, 3), (6144, 4), (8192, 0)] +
                         [(k, 0) for k in (8, 64, 72, 128, 136, 320, 384, 520, 1032)])
def test_streaming_tiles_start_at_any_slab(name, rounding, storage, eps, k, split_k):
    print(f"{name} k {k} split_k {split_k}", flush=True)
    gs = np.array([1, 16, 0, 64, 65, 128, 3, 40, 17, 100, 2, 129], np.int32)  # single row tiles of both routines, and one that is no such tile
    n, g, m, poisoned = 1032, len(gs), int(gs.sum()), 3
    rng = np.random.default_rng(k)
    r = lambda a: oracle.round_to(a, rounding)
    x, A = r(rng.standard_normal((m, k), np.float32)), r(rng.standard_normal((g, n, k), np.float32) / np.float32(np.sqrt(k)))
    first = int(gs[:poisoned].sum())
    x_in, A_in = x.copy(), A.copy()
    x_in[first:first + gs[poisoned]], A_in[poisoned] = np.nan, np.nan
    y = util.to_np(ops._gmm_fwd(_dev(x_in, storage), _dev(A_in, storage), torch.from_numpy(gs).cuda(), trans_rhs=True, compute_dtype=None,
                                plan=_capi.Plan(_vid(name), split_k=split_k), **HP))
    ref = oracle.gmm(x, np.swapaxes(A, 1, 2), gs, out_dtype="float32", acc=np.float64)
    live = np.ones(m, bool)
    live[first:first + gs[poisoned]] = False
    assert np.all(np.isnan(y[~live]))
    err = np.linalg.norm(y[live] - ref[live], axis=1) / np.linalg.norm(ref[live], axis=1)
    assert err.max() < eps + k * 2.0 ** -24, err.max()  # one rounding of the result on top of fp32 sums of k products


@pytest.mark.parametrize("name,rounding,storage,eps", CORES)
def test_a_rows_bits_do_not_depend_on_the_groups_before(name, rounding, storage, eps):
    """The same rows and weights of the last group behind groups of other sizes, with more and with fewer row tiles: the same bits,
    as long as no tile is cut along K."""
    k, n, rows = 2048, 264, 48
    rng = np.random.default_rng(11)
    x_last, A = _dev(rng.normal(size=(rows, k)), storage), _dev(rng.normal(size=(4, n, k)) / np.sqrt(k), storage)
    got = []
    for before in ([16, 0, 100], [300, 1, 100], [1, 1, 1], [0, 0, 0], [700, 300, 257]):
        gs = np.array(before + [rows], np.int32)
        print(f"{name} sizes {gs}", flush=True)
        x = torch.cat([_dev(rng.normal(size=(sum(before), k)), storage), x_last])
        y = ops._gmm_fwd(x, A, torch.from_numpy(gs).cuda(), trans_rhs=True, compute_dtype=None, plan=_capi.Plan(_vid(name), split_k=-1), **HP)
        got.append(y[sum(before):].clone())
    for y in got[1:]:
        assert torch.equal(y.view(torch.int16), got[0].view(torch.int16))
