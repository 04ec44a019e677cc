"""The core of rd_gemm_ws.h on weights beyond the last-level cache, whose short groups it streams: every tile that has such a
kernel, both layouts, groups of one row tile and of several in one launch, against float32 products of each group, and bit for bit
against the same rows and weights in a call with fewer groups, which does not stream."""

import ctypes

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi

pytestmark = pytest.mark.gpu

VARIANTS = [(v.id, v.name.decode(), v.dtype) for v in _capi.variants() if v.name.decode().startswith(("v", "hv"))]
TYPES = {_capi.RD_DTYPE_BF16: (torch.bfloat16, 2.0 ** -8), _capi.RD_DTYPE_F16: (torch.float16, 2.0 ** -11)}


def _gmm(vid, dtype, x, w, gs, n, trans_rhs, split_k):
    (m, k), g = x.shape, w.shape[0]
    plan = _capi.Plan(vid, split_k=split_k)
    ws = torch.empty(_capi.lib.rd_gmm_workspace_bytes(m, g, ctypes.byref(plan)), dtype=torch.uint8, device="cuda")
    y = torch.full((m, n), float("nan"), dtype=x.dtype, device="cuda")
    _capi.check(_capi.lib.rd_gmm(torch.cuda.current_stream().cuda_stream, x.data_ptr(), w.data_ptr(), gs.data_ptr(), y.data_ptr(),
                                 m, k, n, g, int(trans_rhs), dtype, ctypes.byref(plan), ws.data_ptr(), ws.numel()))
    return y


@pytest.mark.parametrize("trans_rhs", [False, True], ids=["nn", "nt"])
@pytest.mark.parametrize("vid,vname,dtype", VARIANTS, ids=[v[1] for v in VARIANTS])
# rows of the weights: whole lines with a contraction that is no whole slab, or a last column tile of 64 columns; cut along K; no
# whole lines, where nothing is streamed
@pytest.mark.parametrize("k,n,split_k", [(1032, 2112, -1), (1088, 2048, -1), (3648, 704, 2), (1048, 2072, -1)])
def test_streamed_weights(vid, vname, dtype, k, n, split_k, trans_rhs):
    if trans_rhs:
        k, n = n, k
    print(f"{vname} k {k} n {n} split_k {split_k} trans_rhs {trans_rhs}", flush=True)
    storage, eps = TYPES[dtype]
    sizes = [16, 0, 64, 65, 1, 128, 129, 33, 300, 2] + [7] * 64
    g, m, few = len(sizes), sum(sizes) + 3, 10
    assert 2 * g * k * n >= 300e6 and m < 128 * g and 2 * few * k * n < 300e6
    gen = torch.Generator(device="cuda")
    gen.manual_seed(k)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda", dtype=storage)
    x, w = rand(m, k), rand(g, *((n, k) if trans_rhs else (k, n))).mul_(k ** -0.5)
    gs = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    y = _gmm(vid, dtype, x, w, gs, n, trans_rhs, split_k)
    row = 0
    for i, rows in enumerate(sizes):
        wi = (w[i].T if trans_rhs else w[i]).float().contiguous()
        ref = x[row:row + rows].float() @ wi
        err = (y[row:row + rows].float() - ref).norm(dim=1) / ref.norm(dim=1)
        # one rounding of the result on top of two float32 sums of k products
        assert rows == 0 or float(err.max()) < eps + 2 * k * 2.0 ** -24, (i, float(err.max()))
        row += rows
    assert not y[row:].any()
    if split_k < 0:
        head = int(np.sum(sizes[:few]))
        alone = _gmm(vid, dtype, x[:head], w[:few], gs[:few].clone(), n, trans_rhs, split_k)
        assert torch.equal(alone.view(torch.int16), y[:head].view(torch.int16))
