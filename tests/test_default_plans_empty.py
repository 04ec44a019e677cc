"""Plans for products without rows, groups, contraction or columns: the library names a tile that takes the call, and the product runs."""

import itertools

import pytest
import torch

import gpu_ragged_dot_amd as rd
from gpu_ragged_dot_amd import _capi, planner

DTYPES = range(_capi.RD_DTYPE_BF16, _capi.RD_DTYPE_F16 + 1)
OPS = (_capi.OP_GMM, _capi.OP_GMM_TRANS, _capi.OP_TGMM)
SIZES = [(0, 12), (64, 0), (0, 0), (0, 1)]
PITCHES = [(1001, 1515), (1008, 1520), (4097, 333), (4096, 4096), (0, 1515), (1001, 0), (7, 5), (64, 96)]


@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("dtype", DTYPES)
def test_default_plan_of_an_empty_product(dtype, aligned):
    variants = _capi.variants()
    for op, (m, g), (k, n) in itertools.product(OPS, SIZES, PITCHES):
        plan = _capi.default_plan(op, m, k, n, g, dtype, aligned)
        assert variants[plan.variant].dtype == dtype, (op, m, k, n, g)
        assert not variants[plan.variant].vec or (aligned and k % 8 == 0 and n % 8 == 0)


def test_selected_plan_of_an_empty_batch():
    for op in OPS:
        assert planner.select_plan(op, 0, 1001, 1515, 8).variant >= 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k,n", [(1001, 1515), (4097, 333), (1008, 1520)])
def test_empty_batch(k, n, dtype):
    x = torch.zeros(0, k, dtype=dtype, device="cuda", requires_grad=True)
    A = torch.ones(3, k, n, dtype=dtype, device="cuda", requires_grad=True)
    sizes = torch.zeros(3, dtype=torch.int32, device="cuda")
    y = rd.ragged_dot(x, A, sizes)
    assert y.shape == (0, n)
    y.sum().backward()
    assert x.grad.shape == (0, k) and A.grad.shape == A.shape and not A.grad.any()
