"""tgmm into a dA whose rows are no whole number of 128-byte lines, against the oracle."""

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi
from oracle import ragged_dot_oracle as oracle
from tests import util

gpu = pytest.mark.gpu


def _dev(a, storage):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda().to(storage)


TGMM_VARIANTS = [(v.id, v.name.decode()) for v in _capi.variants()
                 if v.dtype == _capi.RD_DTYPE_BF16 and v.direct_to_lds and _capi.lib.rd_variant_takes(v.id, _capi.OP_TGMM, 512, 256, 256, v.dtype) == _capi.RD_OK]


@gpu
@pytest.mark.parametrize("vid,vname", TGMM_VARIANTS, ids=[v[1] for v in TGMM_VARIANTS])
@pytest.mark.parametrize("k,n", [(128, 8), (136, 264), (264, 336), (256, 528)])
def test_rows_that_are_no_whole_lines(vid, vname, k, n):
    """dA with rows of a multiple of 16 bytes, not of 128: groups around the row count up to which the lines at a tile's edges
    are stored apart, every element written once and nothing written outside dA."""
    print(f"edge lines, variant {vname} k {k} n {n}", flush=True)
    gs = np.array([1, 80, 81, 0, 17, 200], np.int32)
    g, m = len(gs), int(gs.sum())
    rng = np.random.default_rng(n)
    r = lambda a: oracle.round_to(a, "bfloat16")
    x, dy = r(rng.normal(size=(m, k))), r(rng.normal(size=(m, n)))
    guard = 64
    for shift in (0, 8):  # dA on a 128-byte line or 16 bytes past one
        buf = torch.full((guard + shift + g * k * n + guard,), float("nan"), dtype=torch.bfloat16, device="cuda")
        dA = buf[guard + shift:guard + shift + g * k * n].view(g, k, n)
        ws = torch.empty(_capi.lib.rd_tgmm_workspace_bytes(m, g, None), dtype=torch.uint8, device="cuda")
        xs, dys, gst, plan = _dev(x, torch.bfloat16), _dev(dy, torch.bfloat16), torch.from_numpy(gs).cuda(), _capi.Plan(vid)
        _capi.check(_capi.lib.rd_tgmm(torch.cuda.current_stream().cuda_stream, xs.data_ptr(), dys.data_ptr(), gst.data_ptr(), dA.data_ptr(),
                                      m, k, n, g, _capi.RD_DTYPE_BF16, plan, ws.data_ptr(), ws.numel()))
        ref = oracle.tgmm(x, dy, gs, out_dtype="float32", acc=np.float64)
        got = util.to_np(dA)
        for i in range(g):
            # every element: half a unit in the last place of bf16, and fp32 sums of at most 200 products of N(0, 1) values
            assert np.all(np.abs(got[i] - ref[i]) <= 2.0 ** -8 * np.abs(ref[i]) + 200 * 2.0 ** -24 * 16), f"dA[{i}] shift {shift}"
        assert torch.isnan(buf[:guard + shift]).all() and torch.isnan(buf[guard + shift + g * k * n:]).all()
