"""f16 products of short prompts: the kernel for at most 16 rows, and the row heights of the 64-column tiles that keep a product
(or w1 and w3 in one pass) in one round of workgroups.  The kernel for at most 160 rows takes many of these sizes (test_gpu_rows_products.py); GEMM_ROWS=0
keeps it away where another one is meant."""
import numpy as np
import pytest

from common import Shape, make_gpu, make_oracle, max_rel_err, options, synth_weights
from rllama_amd import Tensor

pytestmark = pytest.mark.gpu
TOL_F16 = 1e-2  # relative, as the other whole-model tests: f16 rounding decisions flip with the order of sums


def _f16(rng, rows, cols, std):
    return (rng.standard_normal((rows, cols)) * std).astype(np.float16)


def _exact(a, b):
    """The float64 product and how far an f16-rounded fp32 sum may lie from it: half a unit in the last place of f16, and k / 16 + 16
    additions that round (or truncate) to 2^-23 of a partial sum bounded by sum |a| |b|."""
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    exact = a64 @ b64.T
    noise = (np.abs(a64) @ np.abs(b64).T) * ((a.shape[1] / 16 + 16) * 2.0 ** -23)
    return exact, 0.5 * _ulp(np.abs(exact) + noise) + noise


def _ulp(x):
    return np.spacing(np.maximum(x, 2.0 ** -14).astype(np.float16)).astype(np.float64)


def _check(got, a, b):
    exact, tol = _exact(a, b)
    assert np.all(np.abs(got.astype(np.float64) - exact) <= tol)


def _check_gate(got, a, w1, w3):
    """f16(silu(g) u) with g and u off by their tolerances: |silu'| <= 1.1, so |u| 1.1 dg + |silu(g)| du + 1.1 dg du, 1e-6 of the value for
    the hardware exponential and reciprocal, and the last rounding."""
    (g, dg), (u, du) = _exact(a, w1), _exact(a, w3)
    silu = g / (1.0 + np.exp(-g))
    tol = np.abs(u) * 1.1 * dg + np.abs(silu) * du + 1.1 * dg * du + 1e-6 * np.abs(silu * u)
    assert np.all(np.abs(got.astype(np.float64) - silu * u) <= tol + 0.5 * _ulp(np.abs(silu * u) + tol))


# k: two K-steps for each of sixteen wavefronts, a remainder, bursts and a remainder, just below the kernel's range; columns: less than a tile, a remainder, and more tiles than
# the part has compute units once (8 wavefronts) and twice (4 wavefronts, at most 8 rows)
@pytest.mark.parametrize("m,n,k", [(2, 8, 1024), (16, 40, 1056), (7, 4099, 1120), (15, 8216, 1088), (8, 8216, 1088), (16, 1024, 2080), (9, 2048, 2816), (5, 200, 992)])
def test_product_of_few_rows(ctx, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, b = _f16(rng, m, k, 1.0), _f16(rng, n, k, 0.05)
    A, B = Tensor.from_numpy(ctx, a), Tensor.from_numpy(ctx, b)
    _check(A.matrix_mul_transposed(B).to_numpy(), a, b)
    if n % 8 == 0:
        w3 = _f16(rng, n, k, 0.05)
        _check_gate(A.ffn_gate(B, Tensor.from_numpy(ctx, w3)).to_numpy(), a, b, w3)


# long rows, tiles that make one round and a half with bursts that are not whole, columns for more than three rounds
@pytest.mark.parametrize("m,n,k", [(16, 2048, 5632), (2, 1024, 11008), (12, 6144, 2560), (8, 16384, 1408), (8, 5120, 1280), (3, 2048, 6912)])
def test_few_rows_that_the_tiled_kernels_do_better(ctx, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, b = _f16(rng, m, k, 1.0), _f16(rng, n, k, 0.05)
    A, B = Tensor.from_numpy(ctx, a), Tensor.from_numpy(ctx, b)
    with options(ctx, GEMM_ROWS="0"):
        got = A.matrix_mul_transposed(B).to_numpy()
    _check(got, a, b)
    with options(ctx, GEMM_ROWS="0", GEMM_SKINNY="0"):
        assert np.array_equal(got, A.matrix_mul_transposed(B).to_numpy())


def test_two_products_of_few_rows_on_more_workgroups_than_compute_units(ctx):
    rng = np.random.default_rng(95)
    a, w1, w3 = _f16(rng, 16, 2048, 1.0), _f16(rng, 5632, 2048, 0.05), _f16(rng, 5632, 2048, 0.05)
    A, W1, W3 = (Tensor.from_numpy(ctx, t) for t in (a, w1, w3))
    with options(ctx, GEMM_ROWS="0"):
        got = A.ffn_gate(W1, W3).to_numpy()
    _check_gate(got, a, w1, w3)
    with options(ctx, GEMM_ROWS="0", GEMM_SKINNY="0"):
        assert np.array_equal(got, A.ffn_gate(W1, W3).to_numpy())


# 17 heads of 64: K that only this kernel takes
@pytest.mark.parametrize("dim,heads,ffn", [(1024, 16, 2816), (1024, 8, 1024), (1024, 64, 1056), (1088, 17, 2880)])
@pytest.mark.parametrize("n", [2, 15, 16, 17])
@pytest.mark.parametrize("rows", ["1", "0"])
def test_prompt_of_few_rows(ctx, dim, heads, ffn, n, rows):
    """A whole prompt and the token behind it, head dimensions 64, 128 and 16: residual, SiLU-gate and RoPE / cache / V^T epilogues."""
    shape = Shape(dim=dim, n_layers=2, n_heads=heads, ffn_hidden=ffn, vocab_size=64, max_seq_len=80)
    W = synth_weights(shape, seed=91, std=0.05, norm_ones=False)
    toks = np.random.default_rng(92).integers(0, shape.vocab_size, 71)
    om, gm = make_oracle(shape, W, True), make_gpu(ctx, shape, W, True)
    gc, oc = gm.make_caches(), om.make_caches()
    with options(ctx, GEMM_ROWS=rows):
        gm.forward(toks[:70], 0, gc)  # leaves other rows' values in the work buffers
        gc = gm.make_caches()
        assert max_rel_err(gm.forward(toks[:n], 0, gc), om.forward(toks[:n], 0, oc)) < TOL_F16
        assert max_rel_err(gm.forward(toks[n:n + 1], n, gc), om.forward(toks[n:n + 1], n, oc)) < TOL_F16
    gm.free()


# 44 column tiles: row tiles of 32 up to 160 rows, of 64 to 320, of 128 to 640, of 192 to 960, of 256 to 1280; 16 and 48 column tiles
@pytest.mark.parametrize("m,n,k", [(33, 2816, 1024), (160, 2816, 1088), (161, 2816, 1024), (321, 2816, 512), (641, 2816, 512), (961, 2816, 576), (600, 1024, 2816),
                                   (40, 1024, 2816), (130, 3072, 3072), (300, 3000, 1024)])
def test_lowest_row_tile_in_one_round(ctx, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, b, w3 = _f16(rng, m, k, 1.0), _f16(rng, n, k, 0.05), _f16(rng, n, k, 0.05)
    A, B, W3 = (Tensor.from_numpy(ctx, t) for t in (a, b, w3))
    with options(ctx, GEMM_ROWS="0"):
        _check(A.matrix_mul_transposed(B).to_numpy(), a, b)
    got = A.ffn_gate(B, W3).to_numpy()
    with options(ctx, GEMM_DUAL="1"):  # another tile, the same order of additions
        assert np.array_equal(got, A.ffn_gate(B, W3).to_numpy())


@pytest.mark.parametrize("m,n,k,cut", [(131, 1024, 8192, True), (400, 1024, 5184, True), (131, 1024, 5120, False), (131, 704, 8192, False)])
def test_two_products_of_long_rows_are_cut(ctx, m, n, k, cut):
    rng = np.random.default_rng(m + n)
    A, W1, W3 = (Tensor.from_numpy(ctx, _f16(rng, r, k, std)) for r, std in ((m, 1.0), (n, 0.02), (n, 0.02)))
    got = A.ffn_gate(W1, W3).to_numpy()
    same = {}
    for mode in ("0", "3"):  # two launches, cut along K; one pass, whole sums
        with options(ctx, GEMM_DUAL=mode):
            same[mode] = np.array_equal(got, A.ffn_gate(W1, W3).to_numpy())
    assert same == {"0": cut, "3": not cut}


# wq|wk|wv, wo and w2 of whole prompts on the narrow tiles: dim 1024 has 48, 16 and 16 column tiles (row tiles of 32 up to 160 and 512 rows, of
# 64 up to 320 and 1024, of 128 up to 640), 2048 has 96 and 32, 3072 has 144 and 48.  RoPE, cache rows and V^T over several row tiles, the
# residual, and the RMSNorm as a launch of its own; head dimensions 64, 128, 16 and 32
@pytest.mark.parametrize("dim,heads,ffn,rows", [(1024, 16, 2816, (33, 100, 161, 330, 600)), (1024, 32, 1024, (70, 200)), (1024, 64, 1056, (97,)),
                                                (2048, 16, 1024, (40, 81, 130)), (3072, 24, 1024, (33, 70))])
def test_prompt_on_narrow_tiles(ctx, dim, heads, ffn, rows):
    shape = Shape(dim=dim, n_layers=2, n_heads=heads, ffn_hidden=ffn, vocab_size=64, max_seq_len=640)
    W = synth_weights(shape, seed=93, std=0.05, norm_ones=False)
    toks = np.random.default_rng(94).integers(0, shape.vocab_size, 640)
    om, gm = make_oracle(shape, W, True), make_gpu(ctx, shape, W, True)
    for n in rows:
        gc, oc = gm.make_caches(), om.make_caches()
        with options(ctx, GEMM_ROWS="0"):
            assert max_rel_err(gm.forward(toks[:n], 0, gc), om.forward(toks[:n], 0, oc)) < TOL_F16, n
        assert max_rel_err(gm.forward(toks[n:n + 1], n, gc), om.forward(toks[n:n + 1], n, oc)) < TOL_F16, n
    gm.free()
