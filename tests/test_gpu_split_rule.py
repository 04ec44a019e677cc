"""The cut of a launch's last round along K where the plan leaves it to the library: which launches of the 256 x 256 cores are cut, in how many pieces - read
from the arrival counters in the workspace - and that the sums are those of the uncut launch but for the order they are added up in."""

import ctypes

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi

pytestmark = pytest.mark.gpu

TYPES = {_capi.RD_DTYPE_BF16: torch.bfloat16, _capi.RD_DTYPE_F16: torch.float16, _capi.RD_DTYPE_F8E4M3_BF16: torch.float8_e4m3fn}
CORES = [(v.id, v.name.decode(), v.dtype) for v in _capi.variants() if v.dtype in TYPES and v.direct_to_lds and v.tile_m == 256 and v.tile_n == 256]
# group sizes, n, contraction in units of a bfloat16 loop's work (float8: twice the indices), tiles in the last round, pieces of each:
# four row tiles and three column tiles, one round; 67 row tiles and four column tiles, a round and 12
ONE_ROUND, MORE = [300, 200, 17], [60 * 256, 7 * 256 - 100]
CASES = [(ONE_ROUND, 528, 1008, 12, 1), (ONE_ROUND, 528, 1024, 12, 2), (ONE_ROUND, 528, 1504, 12, 2), (ONE_ROUND, 528, 3000, 12, 4), (MORE, 1008, 1504, 12, 1),
         (MORE, 1008, 3000, 12, 4)]


@pytest.mark.parametrize("trans_rhs", [0, 1])
@pytest.mark.parametrize("sizes,n,work,tiles,parts", CASES)
@pytest.mark.parametrize("vid,vname,dtype", CORES, ids=[c[1] for c in CORES])
def test_default_cut(vid, vname, dtype, sizes, n, work, tiles, parts, trans_rhs):
    float8 = dtype == _capi.RD_DTYPE_F8E4M3_BF16
    k = 2 * work if float8 and work > 1024 else work
    if float8 and sizes is ONE_ROUND:  # (no piece is shorter than 512 indices of either type)
        parts = {1024: 1, 1504: 3}.get(work, parts)
    print(f"cut of the last round, {vname} k {k} n {n} groups {sizes} trans_rhs {trans_rhs}", flush=True)
    g, m = len(sizes), sum(sizes) + 9
    gen = torch.Generator(device="cuda").manual_seed(k + n)
    x = torch.randn((m, k), generator=gen, device="cuda").to(TYPES[dtype])
    A = (torch.randn((g, n, k) if trans_rhs else (g, k, n), generator=gen, device="cuda") / (1 if float8 else k ** 0.5)).to(TYPES[dtype])
    gs = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    U = -(-m // 256) + g
    at = -(-((g + 3 * U + 1) * 4) // 256) * 64  # the counters follow the map
    outs = []
    for split_k in (0, -1) + ((parts,) if parts > 1 else ()):
        plan = _capi.Plan(vid, split_k=split_k)
        ws = torch.full((_capi.lib.rd_gmm_workspace_bytes(m, g, ctypes.byref(_capi.Plan(vid))),), 0xA5, dtype=torch.uint8, device="cuda")
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16 if float8 else TYPES[dtype], device="cuda")
        _capi.check(_capi.lib.rd_gmm(torch.cuda.current_stream().cuda_stream, x.data_ptr(), A.data_ptr(), gs.data_ptr(), y.data_ptr(), m, k, n, g, trans_rhs, dtype,
                                     ctypes.byref(plan), ws.data_ptr(), ws.numel()))
        outs.append(y.float())
        if split_k == 0:
            counters = ws.view(torch.int32)[at:at + 256].cpu().numpy()
            arrived = counters[counters != np.int32(-0x5a5a5a5b)]  # (left as they were where no map is built)
            assert np.array_equal(arrived[arrived != 0], [parts] * tiles if parts > 1 else []), arrived
    cut, whole = outs[0], outs[1]
    assert not torch.isnan(cut).any() and not cut[sum(sizes):].any()
    # two roundings of float32 sums that differ by k roundings of the running sum at most
    eps = 2.0 ** -11 if dtype == _capi.RD_DTYPE_F16 else 2.0 ** -8
    assert torch.equal(cut, whole) if parts == 1 else (cut - whole).norm() <= (2 * eps + k * 2.0 ** -24) * whole.norm()
    if parts > 1:
        assert torch.equal(cut, outs[2]) and (float8 or not torch.equal(cut, whole))  # (float8: sums of few bits, exact in any order)
