"""Products of at most 160 (f16) or 96 (fp32) rows on the kernel whose wavefronts split K: plain, cut along K, w1 and w3 in one pass, and inside
prompts of both modes."""
import numpy as np
import pytest

import rllama_amd
from common import Shape, make_gpu, make_oracle, max_rel_err, options, random_f32_weights, synth_weights
from rllama_amd import Tensor
from test_gpu_short_products import TOL_F16, _check, _check_gate, _f16

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx():
    """A context of its own: what these tensors leave in the pool of freed buffers goes with it."""
    c = rllama_amd.Context(0)
    yield c
    c.close()


# rows: every number of 16-row fragments at its first and last row; columns: less than a fragment, a remainder, one round of workgroups on
# two, three and four fragments of columns and a bit; k: one unit of 128, fewer units than stages, odd and even numbers of units, units of 256
# (16 rows from 6144 on), pieces along K of unequal length
@pytest.mark.parametrize("m", [2, 16, 17, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 113, 128, 129, 144, 145, 160])
def test_products(ctx, m):
    rng = np.random.default_rng(m)
    for n, k in ((8, 128), (1000, 256), (24, 640), (4104, 384), (8200, 512), (12296, 256), (16392, 384), (264, 5888), (1032, 6144), (8200, 6144 if m <= 16 else 1152)):
        a, b = _f16(rng, m, k, 1.0), _f16(rng, n, k, 0.05)
        A, B = Tensor.from_numpy(ctx, a), Tensor.from_numpy(ctx, b)
        _check(A.matrix_mul_transposed(B).to_numpy(), a, b)
        if m <= 16 and n <= 8200:
            w3 = _f16(rng, n, k, 0.05)
            _check_gate(A.ffn_gate(B, Tensor.from_numpy(ctx, w3)).to_numpy(), a, b, w3)


def test_what_stays_on_the_other_kernels(ctx):
    """K that is not a multiple of 128, columns that are not a multiple of 8, 161 rows, and the switch."""
    rng = np.random.default_rng(7)
    for m, n, k, same in ((40, 1000, 1088, True), (40, 1004, 1024, True), (161, 1000, 1024, True), (40, 1000, 1024, False)):
        a, b = _f16(rng, m, k, 1.0), _f16(rng, n, k, 0.05)
        A, B = Tensor.from_numpy(ctx, a), Tensor.from_numpy(ctx, b)
        got = A.matrix_mul_transposed(B).to_numpy()
        with options(ctx, GEMM_ROWS="0"):
            want = A.matrix_mul_transposed(B).to_numpy()
        _check(want, a, b)
        assert np.array_equal(got, want) == same


# (rows, columns, K, whether the kernels for any number of rows take it): more than one round of workgroups; cut where their tiles make one round; A beyond an L2;
# each beside sizes on the other side of the line
@pytest.mark.parametrize("m,n,k,other", [(65, 16448, 256, True), (64, 16448, 256, False), (65, 16384, 256, False), (112, 32000, 256, True), (96, 1536, 1536, True),
                                         (64, 1536, 1536, False), (96, 768, 1536, False), (97, 3072, 2560, True), (96, 3072, 2560, False),
                                         (160, 1024, 10752, True), (160, 1024, 10624, False)])
def test_what_the_other_kernels_do_better(ctx, m, n, k, other):
    rng = np.random.default_rng(m + n + k)
    a, b = _f16(rng, m, k, 1.0), _f16(rng, n, k, 0.05)
    A, B = Tensor.from_numpy(ctx, a), Tensor.from_numpy(ctx, b)
    got = A.matrix_mul_transposed(B).to_numpy()
    _check(got, a, b)
    with options(ctx, GEMM_ROWS="0"):
        assert np.array_equal(got, A.matrix_mul_transposed(B).to_numpy()) == other


# whole prompts and the token behind them: residual, SiLU-gate and RoPE / cache / V^T epilogues, whole sums and pieces (ffn 6144), head dimensions
# 16 to 128, V^T read past the last row by the next attention kernel's tiles
@pytest.mark.parametrize("dim,heads,ffn", [(1024, 16, 2816), (1152, 9, 3072), (1024, 64, 1024), (2048, 64, 6144)])
def test_prompts(ctx, dim, heads, ffn):
    shape = Shape(dim=dim, n_layers=2, n_heads=heads, ffn_hidden=ffn, vocab_size=64, max_seq_len=176)
    W = synth_weights(shape, seed=61, std=0.05, norm_ones=False)
    toks = np.random.default_rng(62).integers(0, shape.vocab_size, 176)
    om, gm = make_oracle(shape, W, True), make_gpu(ctx, shape, W, True)
    for n in (3, 16, 17, 47, 64, 79, 96, 111, 128, 129, 160):
        gm.forward(toks, 0, gm.make_caches())  # leaves other rows' values in the work buffers
        gc, oc = gm.make_caches(), om.make_caches()
        assert max_rel_err(gm.forward(toks[:n], 0, gc), om.forward(toks[:n], 0, oc)) < TOL_F16, n
        assert max_rel_err(gm.forward(toks[n:n + 1], n, gc), om.forward(toks[n:n + 1], n, oc)) < TOL_F16, n
    gm.free()


# f32 mode: no rounding points, so only the order of sums differs.  K of an odd number of units of 64 floats, fewer units than stages, pieces along K
# (ffn 6144), column counts that leave a remainder, both products of w1 and w3 on one to four fragments of columns; up to 96 rows and beyond
@pytest.mark.parametrize("dim,heads,ffn", [(64, 2, 192), (192, 3, 520), (1024, 16, 2816), (1088, 17, 2048), (2048, 32, 6144)])
def test_prompts_in_f32_mode(ctx, dim, heads, ffn):
    shape = Shape(dim=dim, n_layers=2, n_heads=heads, ffn_hidden=ffn // 32 * 32, vocab_size=64, max_seq_len=112)
    W = random_f32_weights(shape, seed=63, std=0.7 / dim ** 0.5)
    toks = np.random.default_rng(64).integers(0, shape.vocab_size, 112)
    om, gm = make_oracle(shape, W, False), make_gpu(ctx, shape, W, False)
    for n in (2, 16, 17, 33, 48, 49, 64, 65, 96, 97):
        gm.forward(toks, 0, gm.make_caches())  # leaves other rows' values in the work buffers
        gc, oc = gm.make_caches(), om.make_caches()
        # (the oracle adds in another order too: a few 2^-24 times the square root of K per sum, 1e-6 of the largest logit measured)
        assert max_rel_err(gm.forward(toks[:n], 0, gc), om.forward(toks[:n], 0, oc)) < 1e-5, n
        assert max_rel_err(gm.forward(toks[n:n + 1], n, gc), om.forward(toks[n:n + 1], n, oc)) < 1e-5, n
    gm.free()
