"""float32 tgmm into a dA whose rows are no whole number of 64-byte halves of a line, on every tile of the any-pitch core, against the oracle."""

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi
from oracle import ragged_dot_oracle as oracle
from tests import util

CODES = (_capi.RD_DTYPE_F32, _capi.RD_DTYPE_F32_BF16)
CASES = [(v.id, v.name.decode(), v.dtype, k, n) for v in _capi.variants() if v.dtype in CODES
         for k, n in [(8, 8), (136, 264), (131, 77), (257, 515), (128, 256)]
         if _capi.lib.rd_variant_takes(v.id, _capi.OP_TGMM, 512, k, n, v.dtype) == _capi.RD_OK]


@pytest.mark.gpu
@pytest.mark.parametrize("gs", [[1, 120, 121, 0, 17, 200], [2, 120, 121, 0, 17, 700]], ids=["short", "long"])
@pytest.mark.parametrize("vid,vname,dtype,k,n", CASES, ids=[f"{c[1]}-{c[3]}-{c[4]}" for c in CASES])
def test_rows_that_are_no_whole_halves_of_a_line(vid, vname, dtype, k, n, gs):
    """Groups around the row count up to which such rows are stored plainly, in launches whose groups average at most that and more; every
    element written once and nothing outside dA."""
    print(f"edge lines, variant {vname} k {k} n {n} groups {gs}", flush=True)
    gs = np.array(gs, np.int32)
    g, m = len(gs), int(gs.sum())
    rng = np.random.default_rng(n)
    x, dy = (rng.integers(-2, 3, size=(m, width)).astype(np.float32) for width in (k, n))  # sums of at most 2800: exact
    want = oracle.tgmm(x, dy, gs, out_dtype="float32", acc=np.float64)
    xs, dys, gst, plan = torch.from_numpy(x).cuda(), torch.from_numpy(dy).cuda(), torch.from_numpy(gs).cuda(), _capi.Plan(vid)
    guard = 64
    for shift in (0, 4):  # dA on a 128-byte line or 16 bytes past one
        buf = torch.full((guard + shift + g * k * n + guard,), float("nan"), device="cuda")
        dA = buf[guard + shift:guard + shift + g * k * n].view(g, k, n)
        ws = torch.empty(_capi.lib.rd_tgmm_workspace_bytes(m, g, None), dtype=torch.uint8, device="cuda")
        _capi.check(_capi.lib.rd_tgmm(torch.cuda.current_stream().cuda_stream, xs.data_ptr(), dys.data_ptr(), gst.data_ptr(), dA.data_ptr(),
                                      m, k, n, g, dtype, plan, ws.data_ptr(), ws.numel()))
        assert np.array_equal(util.to_np(dA), want), f"shift {shift}"
        assert torch.isnan(buf[:guard + shift]).all() and torch.isnan(buf[guard + shift + g * k * n:]).all()
