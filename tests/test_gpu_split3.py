"""fp32 products on the bf16 matrix cores (three parts per value): against float64, against the fp32 matrix instruction, and the
values the parts cannot hold."""
import time

import numpy as np
import pytest

from common import options
from rllama_amd import Tensor

pytestmark = pytest.mark.gpu
f32 = np.float32


def _product(ctx, a, b, split3="1"):
    """The product with three parts per value wherever the kernel can run ("1"), on the fp32 instruction ("0") or as the library chooses (None)."""
    with options(ctx, **({} if split3 is None else {"GEMM_SPLIT3": split3})):
        return Tensor.from_numpy(ctx, a).matrix_mul_transposed(Tensor.from_numpy(ctx, b)).to_numpy()


# rows: one to eight 32-row tiles of a workgroup (with both parities of their split between the row groups), remainders, more than
# one row tile; columns: less than, exactly and just over a tile of 128; k: one K-tile, fewer than the stages, cut along K
@pytest.mark.parametrize("m,n,k", [(2, 128, 32), (2, 129, 32), (32, 300, 32), (255, 130, 512), (224, 300, 96), (33, 129, 96), (65, 300, 64), (97, 2816, 160), (128, 4096, 4096), (160, 130, 1184), (192, 384, 352),
                                   (200, 3072, 1024), (255, 64, 512), (257, 515, 2048), (300, 4096, 4096)])
def test_split3_product_against_float64(ctx, m, n, k):
    rng = np.random.default_rng(m * 131 + n)
    a = rng.standard_normal((m, k)).astype(f32)
    b = (rng.standard_normal((n, k)) * 0.02).astype(f32)
    exact = a.astype(np.float64) @ b.astype(np.float64).T
    got = _product(ctx, a, b)
    # 6 products of every 16 values of k are added one after the other, each addition rounded to at most 2^-24 of a partial sum
    # that sum |a| |b| bounds (2^-23: the matrix cores may truncate), plus the parts left out (2^-24) and the pieces' sums (18)
    bound = (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T) * ((6 * k / 16 + 1 + 18) * 2.0 ** -23)
    assert np.all(np.abs(got - exact) <= bound)
    plain = _product(ctx, a, b, "0")
    assert not np.array_equal(got, plain)  # the sums of the two ways differ in their last bits
    err, err_plain = (np.linalg.norm(x - exact) / np.linalg.norm(exact) for x in (got, plain))
    assert err <= max(err_plain, 2.0 ** -24), (err, err_plain)


# short rows, tiles that make whole rounds on the fp32 instruction, and many rows of few columns (1.1 to 1.6 times as fast there); a prompt
# projection, ragged rows and one 32-row tile of weights that the fp32 instruction cuts badly
@pytest.mark.parametrize("m,n,k,parts", [(2, 704, 256, False), (128, 704, 256, False), (400, 3072, 64, False), (24, 1408, 1408, False), (16, 4096, 2048, False),
                                         (1024, 64, 2048, False), (200, 4096, 4096, True), (131, 3000, 1024, True), (8, 5632, 1408, True)])
def test_the_faster_of_the_two_ways_is_taken(ctx, m, n, k, parts):
    rng = np.random.default_rng(m + n)
    a, b = rng.standard_normal((m, k), dtype=f32), rng.standard_normal((n, k), dtype=f32)
    by_parts, plain = _product(ctx, a, b, "1"), _product(ctx, a, b, "0")
    assert not np.array_equal(by_parts, plain)
    assert np.array_equal(_product(ctx, a, b, None), by_parts if parts else plain)


@pytest.mark.parametrize("switch", [{"GEMM_SPLIT_K": "3"}, {"GEMM_TILE": "1"}])
def test_switches_of_the_fp32_instruction_take_effect(ctx, switch):
    rng = np.random.default_rng(12)
    a, b = rng.standard_normal((100, 4096), dtype=f32), rng.standard_normal((3000, 4096), dtype=f32)
    with options(ctx, **switch):
        assert np.array_equal(_product(ctx, a, b, None), _product(ctx, a, b, "0"))


def test_split3_product_with_infinities_nan_and_the_largest_values(ctx):
    rng = np.random.default_rng(5)
    m, n, k = 40, 3072, 256
    a = rng.standard_normal((m, k)).astype(f32)
    b = rng.standard_normal((n, k)).astype(f32)
    a[3, 5], a[7, 9], a[11, 1], a[21, 3] = np.inf, -np.inf, np.nan, np.finfo(f32).max   # the parts cannot hold the last
    b[50, 200], b[51, 5], b[60], b[70, 3] = np.inf, 0.0, 0.0, 1e-30
    b[:, 3] *= f32(0.125)                                                                 # FLT_MAX times this stays finite ...
    b[2000:, 3] *= f32(1000.0)                                                            # ... or overflows
    with np.errstate(all="ignore"):
        want = (a.astype(np.float64) @ b.astype(np.float64).T).astype(f32)
    got = _product(ctx, a, b)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    ok = np.isfinite(want)
    with np.errstate(all="ignore"):
        bound = (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T)[ok] * ((k + 20) * 2.0 ** -23)
    assert np.all(np.abs(got[ok].astype(np.float64) - want[ok]) <= bound)


def test_split3_parts_add_up_to_the_value(ctx):
    """Rows of the unit matrix pick values out of B: the three parts of every fp32 number below 2^112 (larger ones are not taken apart),
    whatever stands beside it, add up to it."""
    rng = np.random.default_rng(9)
    n, k = 3072, 64
    sign, exponent, fraction = (rng.integers(0, top, (n, k), dtype=np.uint32) for top in (2, 127 + 112, 1 << 23))
    b = (sign << 31 | exponent << 23 | fraction).view(f32)
    assert np.array_equal(_product(ctx, np.eye(k, dtype=f32), b), b.T)


# operands down to the smallest fp32 numbers (beside large ones, so that the product is not tiny), and products that are subnormal
@pytest.mark.parametrize("ea,eb", [(-109, 60), (-120, 60), (60, -126), (-140, 60), (60, -145), (-70, -70), (-20, -115)])
def test_split3_product_of_tiny_values(ctx, ea, eb):
    rng = np.random.default_rng(8)
    m, n, k = 33, 3072, 288
    a = (rng.standard_normal((m, k)) * 2.0 ** ea).astype(f32)
    b = (rng.standard_normal((n, k)) * 2.0 ** eb).astype(f32)
    exact = a.astype(np.float64) @ b.astype(np.float64).T
    got = _product(ctx, a, b)
    # the bound of the ordinary values, and half a unit of the smallest fp32 number where the result is one
    bound = (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T) * ((6 * k / 16 + 1 + 18) * 2.0 ** -23) + 2.0 ** -150
    assert np.all(np.abs(got - exact) <= bound)
    if ea + eb > -100 and min(ea, eb) >= -126:  # (operands of few bits: the additions of both ways are nearly exact, neither is ahead)
        plain = _product(ctx, a, b, "0")
        err, err_plain = (np.linalg.norm((x - exact) / np.abs(exact).max()) for x in (got, plain))
        assert err <= err_plain, (err, err_plain)


def test_split3_product_of_nan_is_not_slow(ctx):
    """Elements that are not finite are computed again: that is at most the product on the fp32 instruction (1.5 times this one) with
    loads that are not staged, about 3 times the product in all; a plain loop per element takes 100 times."""
    rng = np.random.default_rng(7)
    m, n, k = 200, 11008, 4096
    b = Tensor.from_numpy(ctx, (rng.standard_normal((n, k), dtype=f32) * f32(0.02)))

    def seconds(a):
        A, times = Tensor.from_numpy(ctx, a), []
        for _ in range(4):
            ctx.sync()
            t = time.perf_counter()
            A.matrix_mul_transposed(b)
            ctx.sync()
            times.append(time.perf_counter() - t)
        return min(times)

    a = rng.standard_normal((m, k), dtype=f32)
    plain = seconds(a)
    a[:, 5] = np.nan
    assert seconds(a) < 20 * plain


@pytest.mark.parametrize("m,n,k", [(1500, 96, 32768), (1537, 96, 40960)])  # the second: rows left after a pass pad to more than the capacity
def test_split3_product_in_passes_over_the_rows(ctx, m, n, k):
    # 6 bytes per element of a: the rows need more than the work memory holds, so they go in several passes
    rng = np.random.default_rng(6)
    a = rng.standard_normal((m, k), dtype=f32)
    b = rng.standard_normal((n, k), dtype=f32)
    exact = a.astype(np.float64) @ b.astype(np.float64).T
    got = _product(ctx, a, b)
    assert np.linalg.norm(got - exact) <= 2e-6 * np.linalg.norm(exact)  # sqrt(6 k / 16) roundings of 2^-24 is 6.6e-6 / 3 when they are independent
