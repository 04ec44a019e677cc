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


TYPES = {_capi.RD_DTYPE_BF16: torch.bfloat16, _capi.RD_DTYPE_F16: torch.float16, _capi.RD_DTYPE_F8E4M3_BF16: torch.float8_e4m3fn}
CASES = [(v.id, v.name.decode(), v.dtype, k, n) for v in _capi.variants() if v.dtype in TYPES and v.direct_to_lds
         for k, n in [(128, 8), (136, 264), (264, 336), (256, 528), (272, 48)]
         if _capi.lib.rd_variant_takes(v.id, _capi.OP_TGMM, 512, k, n, v.dtype) == _capi.RD_OK]


@gpu
@pytest.mark.parametrize("vid,vname,dtype,k,n", CASES, ids=[f"{c[1]}-{c[3]}-{c[4]}" for c in CASES])
@pytest.mark.parametrize("gs", [[1, 80, 81, 0, 17, 200], [1, 80, 81, 0, 17, 400]], ids=["short", "long"])
def test_rows_that_are_no_whole_lines(vid, vname, dtype, k, n, gs):
    """dA with rows of a multiple of 16 bytes, not of 128: groups around the row count up to which the lines at a tile's edges
    are stored apart, in launches whose groups average at most that and more; every element written once and nothing written
    outside dA."""
    print(f"edge lines, variant {vname} k {k} n {n} groups {gs}", flush=True)
    storage = TYPES[dtype]
    gs = np.array(gs, np.int32)
    g, m = len(gs), int(gs.sum())
    rng = np.random.default_rng(n)
    x, dy = (rng.integers(-2, 3, size=(m, width)).astype(np.float32) for width in (k, n))
    guard, out = 64, storage if storage.itemsize == 2 else torch.bfloat16
    for shift in (0, 8):  # dA on a 128-byte line or 16 bytes past one
        buf = torch.full((guard + shift + g * k * n + guard,), float("nan"), dtype=out, device="cuda")
        dA = buf[guard + shift:guard + shift + g * k * n].view(g, k, n)
        ws = torch.empty(_capi.lib.rd_tgmm_workspace_bytes(m, g, None), dtype=torch.uint8, device="cuda")
        xs, dys, gst, plan = _dev(x, storage), _dev(dy, storage), torch.from_numpy(gs).cuda(), _capi.Plan(vid)
        _capi.check(_capi.lib.rd_tgmm(torch.cuda.current_stream().cuda_stream, xs.data_ptr(), dys.data_ptr(), gst.data_ptr(), dA.data_ptr(),
                                      m, k, n, g, dtype, plan, ws.data_ptr(), ws.numel()))
        # whole numbers: every sum of 400 products is exact in float32, so each element is its rounding to the result's type
        want = oracle.round_to(oracle.tgmm(x, dy, gs, out_dtype="float32", acc=np.float64), "float16" if out == torch.float16 else "bfloat16")
        assert np.array_equal(util.to_np(dA), want), f"shift {shift}"
        assert torch.isnan(buf[:guard + shift]).all() and torch.isnan(buf[guard + shift + g * k * n:]).all()
