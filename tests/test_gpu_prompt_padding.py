"""A prompt's result does not depend on what earlier prompts left in the padding of the work buffers."""
import numpy as np
import pytest

import rllama_amd
from common import Shape, make_gpu, options, synth_weights

pytestmark = pytest.mark.gpu


# head dimensions 16 and 32, and 64 with the switch, take the two-product form of attention, whose P.V product reads V^T up to the next
# 128 positions; dim 1024: the few-row kernel (10), tiles of 32 and 64 rows; dim 256: tiles of 128 rows and the cut product, which
# leaves RoPE to a kernel of its own
# f32 mode, whose padding ends at the next 64 positions: head dimensions 32, 64 and 128
@pytest.mark.parametrize("dim,heads,gemm_form,f16", [(1024, 64, False, True), (1024, 32, False, True), (1024, 16, True, True), (256, 16, False, True), (256, 8, False, True),
                                                     (256, 8, False, False), (256, 4, False, False), (256, 2, False, False)])
def test_prompt_after_a_prompt_of_nan(ctx, dim, heads, gemm_form, f16):
    shape = Shape(dim=dim, n_layers=2, n_heads=heads, ffn_hidden=2 * dim, vocab_size=64, max_seq_len=256)
    W = synth_weights(shape, seed=17, std=0.05, norm_ones=False)
    W[(rllama_amd.TOK_EMB, 0)][63] = 0x7E00  # NaN: every key and value of this token
    gm = make_gpu(ctx, shape, W, f16)
    toks = np.random.default_rng(18).integers(0, 63, 256)
    with options(ctx, **({"PREFILL_ATTN": "gemm"} if gemm_form else {})):
        for n in (10, 20, 40, 70, 100, 130, 200):
            want = gm.forward(toks[:n], 0, gm.make_caches())
            assert np.isnan(gm.forward(np.full(256, 63), 0, gm.make_caches())).all()
            got = gm.forward(toks[:n], 0, gm.make_caches())
            assert np.isfinite(want).all() and np.array_equal(got, want), n
    gm.free()
