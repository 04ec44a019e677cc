"""``ragged_dot`` / ``trans_ragged_dot`` with the reference's Python signature, running on HIP kernels.

Mirrors gpu_ragged_dot.py:345-454 (``gmm``, ``tgmm``, their aliases and the custom VJP).  Arrays are
``torch.Tensor`` on a ROCm device: torch supplies device memory, the stream and the autograd engine, nothing else - every
product is computed by ``csrc/libragged_dot_hip.so`` through its C ABI.  What a call does on the host - checks, plan,
allocation, the autograd node - is native code (``csrc/rd_torch.cpp``); this module maps the reference's keywords onto it.
"""

from __future__ import annotations

from typing import Optional

import torch

from . import _capi, _tracing, planner
from ._native import lib as _native
from .planner import CHUNK_M, DEFAULT_BLOCK_K, DEFAULT_BLOCK_M, DEFAULT_BLOCK_N

__all__ = ["gmm", "tgmm", "ragged_dot", "trans_ragged_dot", "ragged_dot_vjp", "make_group_metadata"]

_DTYPES = {torch.bfloat16: _capi.RD_DTYPE_BF16, torch.float32: _capi.RD_DTYPE_F32,
           torch.float8_e4m3fn: _capi.RD_DTYPE_F8E4M3_BF16, torch.float16: _capi.RD_DTYPE_F16}


# (storage dtype, compute_dtype) of the usual calls; _dtype_code() explains the rest
_CODES = {(t, None): code for t, code in _DTYPES.items()}
_CODES.update({(t, t): code for t, code in _DTYPES.items()})
_CODES[torch.float32, torch.bfloat16] = _capi.RD_DTYPE_F32_BF16


def _dtype_code(t: torch.Tensor, compute_dtype, acc_dtype) -> int:
    """Element-type code for the C ABI from the storage dtype and the reference's ``compute_dtype``
    (gpu_ragged_dot.py:116-119, 145: operands are cast to compute_dtype before the dot; None = the storage dtype)."""
    if t.dtype not in _DTYPES:
        raise TypeError(f"unsupported dtype {t.dtype}; operands are bfloat16, float16, float32 or float8_e4m3fn")
    if acc_dtype not in (None, torch.float32):
        raise NotImplementedError("accumulation is always float32 on the matrix cores")
    if t.dtype == torch.float8_e4m3fn:
        if compute_dtype not in (None, torch.bfloat16, torch.float32, torch.float8_e4m3fn):
            raise NotImplementedError(f"no kernel for compute_dtype={compute_dtype} on float8 operands")
        return _capi.RD_DTYPE_F8E4M3_BF16  # float8 products are exact in every one of these types; accumulation is fp32
    if compute_dtype is None or compute_dtype == t.dtype:
        return _DTYPES[t.dtype]
    if t.dtype == torch.float32 and compute_dtype == torch.bfloat16:
        return _capi.RD_DTYPE_F32_BF16  # rounded to bf16 on the way to the bf16 matrix cores, float32 out
    if t.dtype == torch.float16 and compute_dtype == torch.float32:
        return _capi.RD_DTYPE_F16  # as for bfloat16 below: products of float16 values are exact in fp32
    if t.dtype == torch.bfloat16 and compute_dtype == torch.float32:
        # widening bf16 operands changes nothing: their products are exact in fp32 and accumulation is fp32 anyway
        return _capi.RD_DTYPE_BF16
    raise NotImplementedError(f"no kernel for compute_dtype={compute_dtype} on {t.dtype} operands")


def _group_sizes_i32(group_sizes, dev: torch.device) -> torch.Tensor:
    gs = torch.as_tensor(group_sizes)
    if gs.dtype != torch.int32:
        gs = gs.to(torch.int32)
    return gs.to(dev).contiguous()


def _stream_ptr(dev: torch.device) -> int:
    return torch.cuda.current_stream(dev).cuda_stream


def _group_offset(group_offset) -> int:
    """``group_offset`` as a host integer (None = 0; a one-element tensor is read back, which synchronises)."""
    if group_offset is None:
        return 0
    if isinstance(group_offset, torch.Tensor):
        assert group_offset.numel() == 1, "group_offset holds one group index"
        return int(group_offset.item())
    return int(group_offset)


def _aligned16(*tensors: torch.Tensor) -> bool:
    """The fast tile shapes move 16 bytes at a time: every buffer must start on a 16-byte boundary (a view at an odd
    element offset does not, however contiguous it is; what is not contiguous is copied to one that does)."""
    return all(t.data_ptr() % 16 == 0 or not t.is_contiguous() for t in tensors)


def _fields(plan: _capi.Plan) -> tuple:
    return (plan.variant, plan.group_m, plan.group_n, plan.decode_nb, plan.split_k)


def _host_args(x, group_sizes, interpret, compute_dtype, acc_dtype, group_offset):
    """What both products need from the reference's keywords: the element-type code, group_sizes as a tensor, and the first
    group as a host integer (-1: no group_offset given)."""
    if interpret:
        raise NotImplementedError("interpret=True (Pallas interpreter) has no counterpart; kernels run on the GPU only")
    code = _CODES.get((x.dtype, compute_dtype)) if acc_dtype is torch.float32 else None
    if code is None:
        code = _dtype_code(x, compute_dtype, acc_dtype)
    return code, _sizes(group_sizes), -1 if group_offset is None else _group_offset(group_offset)


def _sizes(group_sizes) -> torch.Tensor:
    return group_sizes if isinstance(group_sizes, torch.Tensor) else torch.as_tensor(group_sizes)


def _default_blocks(block_m, block_k, block_n) -> bool:
    return block_m == DEFAULT_BLOCK_M and block_k == DEFAULT_BLOCK_K and block_n == DEFAULT_BLOCK_N


def _select(products, blocks, aligned, operands) -> tuple:
    """Plans of a product, the first of ``products``, and of its gradients if an operand asks for them."""
    wanted = products if torch.is_grad_enabled() and any(t.requires_grad for t in operands) else products[:1]
    return tuple(_fields(planner.select_plan(*p, aligned=aligned or i > 0, **blocks)) for i, p in enumerate(wanted))


def _gmm_plans(x, A, trans_rhs, g, code, block_m, block_k, block_n):
    """Plans for explicit block sizes (gpu_ragged_dot.py:194-197)."""
    (m, k), n = x.shape, A.shape[-2 if trans_rhs else -1]
    planner.normalize_gmm_blocks(block_m, block_k, block_n, m, k, n)  # validates the request
    blocks = dict(block_m=block_m, block_k=block_k, block_n=block_n, dtype=code)
    fwd, bwd = (_capi.OP_GMM_TRANS, _capi.OP_GMM) if trans_rhs else (_capi.OP_GMM, _capi.OP_GMM_TRANS)
    weights = (n, k) if trans_rhs else (k, n)
    return _select(((fwd, m, k, n, g), (bwd, m, n, k, g), (_capi.OP_TGMM, m, *weights, g)), blocks, _aligned16(x, A), (x, A))


def _tgmm_plans(x, y, g, code, block_m, block_k, block_n):
    """The same for tgmm (gpu_ragged_dot.py:308-314)."""
    (m, k), n = x.shape, y.shape[-1]
    planner.normalize_tgmm_blocks(block_m, block_k, block_n, m, k, n)
    blocks = dict(block_m=block_m, block_k=block_k, block_n=block_n, dtype=code)
    return _select(((_capi.OP_TGMM, m, k, n, g), (_capi.OP_GMM_TRANS, m, n, k, g), (_capi.OP_GMM, m, k, n, g)), blocks,
                   _aligned16(x, y), (x, y))


def _gmm(x, A, group_sizes, block_m, block_k, block_n, trans_rhs, interpret, compute_dtype, acc_dtype, chunk_m,
         plan: Optional[_capi.Plan] = None, group_offset=None) -> torch.Tensor:
    """gpu_ragged_dot.py:171-228 (_gpu_gmm_fwd), as an autograd node where an operand asks for it.

    ``group_offset`` (jax.lax.ragged_dot's parameter; not in the reference): A holds the groups
    [group_offset, group_offset + A.shape[0]) of the ones group_sizes describes; rows of the others come out zero."""
    if _tracing.active():
        return _tracing.record(lambda x, A, gs: _gmm(x, A, gs, block_m, block_k, block_n, trans_rhs, interpret, compute_dtype,
                                                     acc_dtype, chunk_m, plan, group_offset), x, A, _sizes(group_sizes))
    code, gs, g_first = _host_args(x, group_sizes, interpret, compute_dtype, acc_dtype, group_offset)
    assert A.ndim == 3 and x.ndim == 2, f"but {A.ndim=} {x.ndim=}"  # :188
    assert chunk_m >= 1 and (group_offset is None or g_first >= 0)
    plans = None
    if plan is not None:
        plans = (_fields(plan),)
    elif not _default_blocks(block_m, block_k, block_n):
        plans = _gmm_plans(x, A, trans_rhs, gs.numel(), code, block_m, block_k, block_n)
    return _native.gmm(x, A, gs, bool(trans_rhs), code, g_first, plans)


def _tgmm(x, y, group_sizes, block_m, block_k, block_n, interpret, compute_dtype, acc_dtype, chunk_m,
          plan: Optional[_capi.Plan] = None, group_offset=None, num_actual_groups=None) -> torch.Tensor:
    """gpu_ragged_dot.py:287-342 (_gpu_tgmm_fwd).  With ``group_offset`` / ``num_actual_groups`` only the slices of the
    groups [group_offset, group_offset + num_actual_groups) are computed: out[i] belongs to group group_offset + i."""
    if _tracing.active():
        return _tracing.record(lambda x, y, gs: _tgmm(x, y, gs, block_m, block_k, block_n, interpret, compute_dtype, acc_dtype,
                                                      chunk_m, plan, group_offset, num_actual_groups),
                               x, y, _sizes(group_sizes))
    del chunk_m  # :303
    code, gs, g_first = _host_args(x, group_sizes, interpret, compute_dtype, acc_dtype, group_offset)
    assert y.ndim == 2 and x.ndim == 2 and x.shape[0] == y.shape[0]  # :304
    assert group_offset is None or g_first >= 0
    plans = None
    if plan is not None:
        plans = (_fields(plan),)
    elif not _default_blocks(block_m, block_k, block_n):
        plans = _tgmm_plans(x, y, gs.numel(), code, block_m, block_k, block_n)
    g_local = -1
    if num_actual_groups is not None:
        g_local = int(num_actual_groups)
        assert g_local >= 1
    return _native.tgmm(x, y, gs, code, g_first, g_local, plans)


def _gmm_fwd(*args, **kw) -> torch.Tensor:
    """The product alone."""
    with torch.no_grad():
        return _gmm(*args, **kw)


def _tgmm_fwd(*args, **kw) -> torch.Tensor:
    with torch.no_grad():
        return _tgmm(*args, **kw)


def gmm(
    x: torch.Tensor,  # [m, k]
    A: torch.Tensor,  # [g, k, n]  ([g, n, k] with trans_rhs)
    group_sizes,  # [g]
    block_m: int = DEFAULT_BLOCK_M,
    block_k: int = DEFAULT_BLOCK_K,
    block_n: int = DEFAULT_BLOCK_N,
    trans_rhs: bool = False,
    interpret: bool = False,
    compute_dtype=None,
    acc_dtype=torch.float32,
    num_warps: Optional[int] = None,
    num_stages: Optional[int] = None,
    chunk_m: int = CHUNK_M,
    group_offset=None,
) -> torch.Tensor:
    """Ragged dot corresponding to jax.lax.ragged_dot: (m, k) x (g, k, n) -> (m, n).  gpu_ragged_dot.py:362-380.

    ``num_warps`` / ``num_stages`` are Triton knobs of the reference and are accepted and ignored; ``chunk_m`` is
    validated only (the kernels split groups by their own tile height).  ``group_offset`` (after the reference's
    parameters; jax.lax.ragged_dot's own keyword): A holds only the groups [group_offset, group_offset + A.shape[0])
    of those in group_sizes - an expert-parallel rank's slice; rows of the other groups are zero.
    """
    del num_warps, num_stages
    if x.dtype == torch.float8_e4m3fn and torch.is_grad_enabled() and (x.requires_grad or A.requires_grad):
        raise NotImplementedError("float8 operands are forward only: their cotangents are bfloat16, differentiate a bfloat16 copy")
    return _gmm(x, A, group_sizes, block_m, block_k, block_n, trans_rhs, interpret, compute_dtype, acc_dtype, chunk_m,
                group_offset=group_offset)


def tgmm(
    x: torch.Tensor,  # [m, k]
    y: torch.Tensor,  # [m, n]
    group_sizes,  # [g]
    block_m: int = DEFAULT_BLOCK_M,
    block_k: int = DEFAULT_BLOCK_K,
    block_n: int = DEFAULT_BLOCK_N,
    interpret: bool = False,
    compute_dtype=None,
    acc_dtype=torch.float32,
    num_warps: Optional[int] = None,
    num_stages: Optional[int] = None,
    chunk_m: int = CHUNK_M,
    group_offset=None,
    num_actual_groups: Optional[int] = None,
) -> torch.Tensor:
    """Transposed ragged dot: (m, k) x (m, n) -> (g, k, n).  gpu_ragged_dot.py:411-428.  With ``group_offset`` /
    ``num_actual_groups`` only the slices of the groups [group_offset, group_offset + num_actual_groups) are computed."""
    del num_warps, num_stages
    return _tgmm(x, y, group_sizes, block_m, block_k, block_n, interpret, compute_dtype, acc_dtype, chunk_m,
                 group_offset=group_offset, num_actual_groups=num_actual_groups)


ragged_dot = gmm  # gpu_ragged_dot.py:406
trans_ragged_dot = tgmm  # gpu_ragged_dot.py:454


def ragged_dot_vjp(x, A, group_sizes, dout, trans_rhs: bool = False, **hp):
    """Forward plus the VJP rule of gpu_ragged_dot.py:383-402 in one call: returns (y, dx, dA)."""
    kw = dict(block_m=DEFAULT_BLOCK_M, block_k=DEFAULT_BLOCK_K, block_n=DEFAULT_BLOCK_N, interpret=False,
              compute_dtype=None, acc_dtype=torch.float32, chunk_m=CHUNK_M)
    kw.update(hp)
    y = _gmm_fwd(x, A, group_sizes, **kw, trans_rhs=trans_rhs)
    dx = _gmm_fwd(dout, A, group_sizes, **kw, trans_rhs=not trans_rhs)
    dA = _tgmm_fwd(x, dout, group_sizes, **kw) if not trans_rhs else _tgmm_fwd(dout, x, group_sizes, **kw)
    return y, dx, dA


def make_group_metadata(group_sizes, m: int, chunk_m: int = CHUNK_M):
    """The scheduling map of gpu_ragged_dot.py:70-90, computed on the device.

    Returns (group_offsets[g], row_it2group[U], row_it2it_in_group[U], total_row_its[1]) as int32 device tensors.
    """
    gs_t = torch.as_tensor(group_sizes)
    if gs_t.device.type != "cuda":
        gs_t = gs_t.to("cuda")
    dev = gs_t.device
    gs = _group_sizes_i32(gs_t, dev)
    g = gs.numel()
    U = _capi.lib.rd_sched_map_len(m, g, chunk_m)
    if U < 0:
        _capi.check(U)
    offs = torch.empty(g, dtype=torch.int32, device=dev)
    t2g = torch.empty(U, dtype=torch.int32, device=dev)
    t2it = torch.empty(U, dtype=torch.int32, device=dev)
    total = torch.empty(1, dtype=torch.int32, device=dev)
    with torch.cuda.device(dev):
        _capi.check(
            _capi.lib.rd_sched_map(_stream_ptr(dev), gs.data_ptr(), g, m, chunk_m, offs.data_ptr(), t2g.data_ptr(),
                                   t2it.data_ptr(), total.data_ptr())
        )
    return offs, t2g, t2it, total
