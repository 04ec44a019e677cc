"""The streaming tiles of trans_rhs begin at slabs of their own (gemm_tile_dlds()): contractions of one slab, around the ring's
depth and with a last slab that is not full, against the oracle."""

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi, ops
from oracle import ragged_dot_oracle as oracle
from tests import util

pytestmark = pytest.mark.gpu

HP = dict(block_m=64, block_k=64, block_n=64, interpret=False, acc_dtype=torch.float32, chunk_m=512)


@pytest.mark.parametrize("name,rounding,storage,eps", [("w256x256x32_w2x2_s5", "bfloat16", torch.bfloat16, 2.0 ** -8),
                                                       ("hw256x256x32_w2x2_s5", "float16", torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("k", [8, 64, 72, 128, 136, 320, 384, 520, 1032, 2048])
def test_streaming_tiles_start_at_any_slab(name, rounding, storage, eps, k):
    print(f"{name} k {k}", flush=True)
    vid = next(v.id for v in _capi.variants() if v.name.decode() == name)
    gs = np.array([1, 16, 0, 64, 65, 128, 3, 40, 17, 100, 2, 129], np.int32)  # single row tiles of both routines, and one that is no such tile
    n, g, m, poisoned = 1032, len(gs), int(gs.sum()), 3
    rng = np.random.default_rng(k)
    r = lambda a: oracle.round_to(a, rounding)
    x, A = r(rng.normal(size=(m, k))), r(rng.normal(size=(g, n, k)) / np.sqrt(k))
    first = int(gs[:poisoned].sum())
    x_in, A_in = x.copy(), A.copy()
    x_in[first:first + gs[poisoned]], A_in[poisoned] = np.nan, np.nan
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().to(storage)
    y = util.to_np(ops._gmm_fwd(dev(x_in), dev(A_in), torch.from_numpy(gs).cuda(), trans_rhs=True, compute_dtype=None,
                                plan=_capi.Plan(vid), **HP))
    ref = oracle.gmm(x, np.swapaxes(A, 1, 2), gs, out_dtype="float32", acc=np.float64)
    live = np.ones(m, bool)
    live[first:first + gs[poisoned]] = False
    assert np.all(np.isnan(y[~live]))
    err = np.linalg.norm(y[live] - ref[live], axis=1) / np.linalg.norm(ref[live], axis=1)
    assert err.max() < eps + k * 2.0 ** -24, err.max()  # one rounding of the result on top of fp32 sums of k products
