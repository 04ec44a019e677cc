"""float32 products as six products of bf16 terms (RsCfg with THREE in csrc/rd_gemm_rs.h): as accurate as products on the float32
instruction at every magnitude, and on that instruction where the terms do not hold the numbers."""

import functools

import numpy as np
import pytest
import torch

from gpu_ragged_dot_amd import _capi, ops

pytestmark = pytest.mark.gpu

HP = dict(block_m=64, block_k=64, block_n=64, interpret=False, compute_dtype=None, acc_dtype=torch.float32, chunk_m=512)
TERMS = ["ft128x256x32_w2x4", "ft128x128x32_w2x4", "ft64x128x32_w2x2"]
WHOLE = "fr64x64x32_w2x2"
CASES = [(name, op) for name in TERMS for op in (0, 1, 2)]


@functools.lru_cache(None)
def variant(name):
    return next(v.id for v in _capi.variants() if v.name.decode() == name)


def product(op, a, b, sizes, name, split_k=0):
    plan = _capi.Plan(variant(name), split_k=split_k)
    a, b, gs = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), torch.tensor(sizes, dtype=torch.int32).cuda()
    if op == 2:
        return ops._tgmm_fwd(a, b, gs, **HP, plan=plan).cpu().numpy()
    return ops._gmm_fwd(a, b, gs, **HP, trans_rhs=op == 1, plan=plan).cpu().numpy()


def operands(op, k, n, sizes, draw):
    m, g = sum(sizes), len(sizes)
    return draw((m, k)), draw((m, n) if op == 2 else (g, n, k) if op == 1 else (g, k, n))


def reference(op, a, b, sizes):
    """The sums and the sums of magnitudes, in float64."""
    out, at = [], 0
    for i, s in enumerate(sizes):
        x, y = a[at:at + s].astype(np.float64), (b[at:at + s] if op == 2 else b[i]).astype(np.float64)
        x, y = (x.T, y) if op == 2 else (x, y.T if op == 1 else y)
        out.append((x @ y, np.abs(x) @ np.abs(y)))
        at += s
    join = np.stack if op == 2 else np.concatenate
    return join([o[0] for o in out]), join([o[1] for o in out])


# edges of tiles and of slabs, odd pitches, a group of one row, an empty one, groups of up to 64 rows behind whole tiles
SHAPES = [(8, 8, [3]), (33, 257, [1, 0, 64, 65]), (64, 128, [127, 129]), (100, 300, [130, 256, 17]), (1027, 385, [321])]


@pytest.mark.parametrize("k,n,sizes", SHAPES)
@pytest.mark.parametrize("name,op", CASES)
def test_every_magnitude(name, op, k, n, sizes):
    rng = np.random.default_rng(k + n)
    # 2^-30 .. 2^30, with zeros: what a term loses of a small number would show beside a large one's zero partner
    def draw(shape):
        v = rng.standard_normal(shape) * np.exp2(rng.integers(-30, 31, shape))
        return np.where(rng.random(shape) < 0.3, 0, v).astype(np.float32)
    a, b = operands(op, k, n, sizes, draw)
    want, magnitudes = reference(op, a, b, sizes)
    got = product(op, a, b, sizes, name)
    length = max(sizes) if op == 2 else k
    # one rounding for every contraction index at most, and the products of terms left out: two of at most 2^-25 of the whole one
    assert (np.abs(got - want) <= (length + 1) * 2.0 ** -24 * magnitudes).all()


@pytest.mark.parametrize("k,n,sizes", SHAPES + [(65, 513, [300, 1, 0, 129]), (200, 250, [128, 127, 200])])
@pytest.mark.parametrize("op", [0, 1])
def test_whole_tiles_of_256_columns(op, k, n, sizes):
    """With the cut off every tile of 128 x 256 is computed whole; otherwise launches of under a round are all halves."""
    rng = np.random.default_rng(k + n + 1)
    a, b = operands(op, k, n, sizes, lambda shape: (rng.standard_normal(shape) * np.exp2(rng.integers(-30, 31, shape))).astype(np.float32))
    want, magnitudes = reference(op, a, b, sizes)
    got = product(op, a, b, sizes, TERMS[0], -1)
    assert (np.abs(got - want) <= (k + 1) * 2.0 ** -24 * magnitudes).all()
    # another group's numbers stay out: loads past a row or a group would bring NaN
    last = len(sizes) - 1
    a[sum(sizes[:last]):], b[last] = np.nan, np.nan
    again = product(op, a, b, sizes, TERMS[0], -1)
    rows = sum(sizes[:last])
    assert np.array_equal(again[:rows], got[:rows]) and np.isnan(again[rows:]).all()


@pytest.mark.parametrize("name,op", CASES)
@pytest.mark.parametrize("low,high", [(0, 0), (-108, 100), (100, -70)])
def test_no_less_accurate_than_the_float32_instruction(name, op, low, high):
    rng = np.random.default_rng(5)
    k, n, sizes = 512, 256, [400, 112]
    a, b = operands(op, k, n, sizes, lambda shape: rng.standard_normal(shape).astype(np.float32))
    a, b = np.ldexp(np.where(np.abs(a) < 0.25, 0.25, a), low), np.ldexp(b, high)  # all above 2^-110
    want, _ = reference(op, a, b, sizes)
    error = [np.linalg.norm(product(op, a, b, sizes, v) - want) for v in (name, WHOLE)]
    assert error[0] <= error[1]


@pytest.mark.parametrize("name", TERMS)
def test_groups_of_few_rows_are_no_less_accurate(name):
    """A product alone is rounded once on the float32 instruction; with few of them what the terms leave out shows."""
    rng = np.random.default_rng(9)
    k, n, few = 256, 512, [1, 2, 3, 4, 5, 6, 8, 12, 16, 24]
    sizes = few + few[::-1]
    a, b = operands(2, k, n, sizes, lambda shape: rng.standard_normal(shape).astype(np.float32))
    want, _ = reference(2, a, b, sizes)
    got, whole = (product(2, a, b, sizes, v) for v in (name, WHOLE))
    for i, rows in enumerate(sizes):
        assert np.linalg.norm(got[i] - want[i]) <= np.linalg.norm(whole[i] - want[i]), rows


@pytest.mark.parametrize("k,n", [(8, 8), (57, 77), (129, 257), (256, 512)])
@pytest.mark.parametrize("name", TERMS)
def test_groups_of_one_and_two_rows_have_the_float32_instructions_bits(name, k, n):
    rng = np.random.default_rng(k)
    sizes = [1, 2, 0, 2, 1, 40, 1, 2]
    a, b = operands(2, k, n, sizes, lambda shape: rng.standard_normal(shape).astype(np.float32))
    a[0, ::3], b[1, ::2], a[3, 1], b[4, 2], a[5, 3], a[46, ::4] = 0, 0, np.inf, np.nan, 1e-40, 2.0 ** -70
    b[46] *= 2.0 ** -60
    got, whole = (product(2, a, b, sizes, v) for v in (name, WHOLE))
    some = [i for i, rows in enumerate(sizes) if rows <= 2]
    assert np.array_equal(got[some].view(np.int32)[~np.isnan(got[some])], whole[some].view(np.int32)[~np.isnan(whole[some])])
    assert np.array_equal(np.isnan(got[some]), np.isnan(whole[some])) and np.isnan(got[some]).any()


@pytest.mark.parametrize("name,op", CASES)
@pytest.mark.parametrize("low,high", [(-50, -50), (-60, -60), (-62, -62), (-63, -63), (-64, -64), (-66, -66), (-70, -50), (-100, -20)])
def test_products_near_the_bottom_of_the_range(name, op, low, high):
    """Products of terms, and from 2^-126 down sums too, below the normal numbers: no less accurate than the float32 instruction."""
    rng = np.random.default_rng(11)
    k, n, sizes = 512, 256, [400, 112]
    a, b = operands(op, k, n, sizes, lambda shape: rng.standard_normal(shape).astype(np.float32))
    a, b = (np.ldexp(np.where(np.abs(v) < 0.25, 0.25, v), by).astype(np.float32) for v, by in ((a, low), (b, high)))
    want, _ = reference(op, a, b, sizes)
    error = [np.linalg.norm((product(op, a, b, sizes, v) - want) * 2.0 ** 100) for v in (name, WHOLE)]  # (norms of squares above 2^-1022)
    assert error[0] <= error[1]


ODD_ONES = [np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 1e-40, 2.0 ** -111, 1e30]


@pytest.mark.parametrize("split_k", [-1, 3])
@pytest.mark.parametrize("odd", ODD_ONES)
@pytest.mark.parametrize("name,op", CASES)
def test_numbers_that_the_terms_do_not_hold(name, op, odd, split_k):
    rng = np.random.default_rng(7)
    k, n, sizes = 1024, 256, [64, 64, 64]
    a, b = operands(op, k, n, sizes, lambda shape: rng.standard_normal(shape).astype(np.float32))
    plain = product(op, a, b, sizes, name, split_k)
    a[70, 1000] = odd  # group 1; in the last piece of a cut
    if odd == 1e30:    # a sum beyond the type's range
        b[70 if op == 2 else 1] *= 1e30
    if op == 2:
        split_k = 0
    got = product(op, a, b, sizes, name, split_k)
    whole = product(op, a, b, sizes, WHOLE, split_k)
    touched, others = (slice(1, 2), [0, 2]) if op == 2 else (slice(64, 128), list(range(64)) + list(range(128, 192)))
    assert np.array_equal(np.isfinite(got), np.isfinite(whole)) and np.array_equal(got[others], plain[others])
    if split_k <= 0 and op != 2:
        assert np.array_equal(got[touched], whole[touched], equal_nan=True)
    else:
        want, magnitudes = reference(op, np.where(np.isfinite(a), a, 0), b, sizes)
        ok = np.isfinite(whole)
        assert (np.abs(got - want) <= 1024 * 2.0 ** -24 * magnitudes)[ok].all()
        assert np.array_equal(got[~ok], whole[~ok], equal_nan=True)


@pytest.mark.parametrize("m,k,n,g", [(3000, 2048, 1111, 5), (1640, 4100, 900, 3), (5000, 300, 2000, 40)])
def test_default_plan(m, k, n, g):
    rng = np.random.default_rng(m)
    p = np.exp(rng.standard_normal(g))
    sizes = rng.multinomial(m - 7, p / p.sum()).tolist()
    for op in (0, 1, 2):
        plan = _capi.default_plan(op, m, k, n, g, _capi.RD_DTYPE_F32)
        name = _capi.variants()[plan.variant].name.decode()
        assert name.startswith("ft")
        a, b = operands(op, k, n, sizes, lambda shape: rng.standard_normal(shape).astype(np.float32))
        want, magnitudes = reference(op, a, b, sizes)
        got = product(op, a, b, sizes, name)
        assert (np.abs(got - want) <= (max(sizes) if op == 2 else k) * 2.0 ** -24 * magnitudes).all()


@pytest.mark.parametrize("k,n", [(8, 8), (57, 77), (65, 257), (225, 131), (321, 72)])
@pytest.mark.parametrize("name,op", CASES)
def test_another_groups_numbers_do_not_reach_a_group(name, op, k, n):
    """Loads that run past a row or a group read NaN there: the other groups' bits stay (a tile that saw one would be computed another way)."""
    rng = np.random.default_rng(k)
    sizes = [257, 0, 1, 63, 40, 129, 7]
    a, b = operands(op, k, n, sizes, lambda shape: rng.standard_normal(shape).astype(np.float32))
    clean = product(op, a, b, sizes, name)
    first, rows = sum(sizes[:4]), sizes[4]
    a[first:first + rows] = np.nan
    if op == 2:
        b[first:first + rows] = np.nan
    else:
        b[4] = np.nan
    got = product(op, a, b, sizes, name)
    hit = np.zeros(len(got), bool)
    hit[4 if op == 2 else slice(first, first + rows)] = True
    assert np.isnan(got[hit]).all() and np.array_equal(got[~hit], clean[~hit])


@pytest.mark.parametrize("k,n,names", [(2048, 56, [WHOLE]), (2048, 128, TERMS), (63, 4000, ["ft64x128x32_w2x2", WHOLE]), (64, 4000, TERMS)])
def test_narrow_and_short_products(k, n, names):
    rng = np.random.default_rng(k)
    sizes = [300, 0, 1700, 1, 999]
    for op in (0, 1):
        name = _capi.variants()[_capi.default_plan(op, sum(sizes), k, n, len(sizes), _capi.RD_DTYPE_F32).variant].name.decode()
        assert name in names
        a, b = operands(op, k, n, sizes, lambda shape: rng.standard_normal(shape).astype(np.float32))
        want, magnitudes = reference(op, a, b, sizes)
        assert (np.abs(product(op, a, b, sizes, name) - want) <= k * 2.0 ** -24 * magnitudes).all()


def test_a_named_tile_is_the_one_that_runs():
    """356 tiles of 128 x 128, the last 100 of them in two pieces, or 178 of 128 x 256, too many to be halved: other sums, whichever the
    library would choose itself."""
    rng = np.random.default_rng(13)
    k, n, sizes = 4096, 512, [89 * 128]
    a, b = operands(0, k, n, sizes, lambda shape: rng.standard_normal(shape).astype(np.float32))
    cut, whole, wide = (product(0, a, b, sizes, name, split_k) for name, split_k in (("ft128x128x32_w2x4", 2), ("ft128x128x32_w2x4", -1), ("ft128x256x32_w2x4", 2)))
    assert not np.array_equal(cut, whole) and np.array_equal(wide, whole)


@pytest.mark.parametrize("m,k,n,g", [(3000, 2048, 1111, 5), (4096, 2048, 2048, 4), (777, 333, 421, 5)])
def test_default_tile_without_pieces(m, k, n, g):
    """split_k = -1 with the library's own tile: the choice counts no halves and no pieces."""
    rng = np.random.default_rng(k)
    sizes = rng.multinomial(m, np.ones(g) / g).tolist()
    a, b = operands(0, k, n, sizes, lambda shape: rng.standard_normal(shape).astype(np.float32))
    want, magnitudes = reference(0, a, b, sizes)
    x, w, gs = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), torch.tensor(sizes, dtype=torch.int32).cuda()
    got = ops._gmm_fwd(x, w, gs, **HP, trans_rhs=False, plan=_capi.Plan(-1, split_k=-1)).cpu().numpy()
    assert (np.abs(got - want) <= k * 2.0 ** -24 * magnitudes).all()
