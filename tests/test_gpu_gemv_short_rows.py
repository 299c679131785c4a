"""Single-row products whose rows are one burst of loads or less: several whole rows per burst, against the walk burst by burst (which the
oracle pins elsewhere) bit for bit: a lane adds its products in the same order either way."""
import numpy as np
import pytest

import oracle
import rllama_amd
from common import Shape, make_gpu, options, synth_weights
from rllama_amd import Tensor

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx():
    """A context of its own: what these tensors leave in the pool of freed buffers goes with it."""
    c = rllama_amd.Context(0)
    yield c
    c.close()


# row lengths around the pieces of 512 halves / 256 floats (1 to 8, and 9, which is walked); rows: fewer than wavefronts of the grid, one
# round of a group and a rest, several groups and a rest
F16_K = (8, 504, 512, 520, 1024, 1032, 1536, 1544, 2048, 2560, 2568, 3072, 3584, 3592, 4096, 4104)
F32_K = (4, 252, 256, 260, 512, 768, 772, 1024, 1280, 1536, 1792, 1796, 2048, 2052)


@pytest.mark.parametrize("f16,k", [(True, k) for k in F16_K] + [(False, k) for k in F32_K])
def test_short_rows_have_the_bits_of_the_walk(ctx, f16, k):
    rng = np.random.default_rng(k)
    for m_rows in (1, 5, 2047, 2049, 8193, 20001 if k <= 1032 else 4100):
        w = (rng.standard_normal((m_rows, k), dtype=np.float32) * 0.05)
        W = Tensor.from_numpy(ctx, oracle.f32_to_f16_bits(w) if f16 else w)
        X = Tensor.from_numpy(ctx, rng.standard_normal((1, k)).astype(np.float32))
        for rx, ry in ((True, True), (False, False)) if f16 else ((False, False),):
            got = W.gemv(X, round_x=rx, round_y=ry).to_numpy()
            with options(ctx, GEMV_BURST="0"):
                want = W.gemv(X, round_x=rx, round_y=ry).to_numpy()
            assert np.array_equal(got, want), (m_rows, rx, ry)


# dims of 1 to 9 pieces (the feed-forward width past the next one), partial last pieces, both modes; the token step from the embedding row to the pick
@pytest.mark.parametrize("dim,ffn,f16", [(64, 520, True), (1024, 2816, True), (1152, 3080, True), (2560, 2200, True), (3584, 2104, True), (4096, 600, True), (4608, 200, True),
                                         (256, 520, False), (576, 1024, False), (1152, 2104, False), (2048, 296, False), (2304, 64, False)])
def test_token_step_of_short_rows(ctx, dim, ffn, f16):
    shape = Shape(dim=dim, n_layers=2, n_heads=dim // 64, ffn_hidden=ffn, vocab_size=4500, max_seq_len=16)
    gm = make_gpu(ctx, shape, synth_weights(shape, seed=3, std=0.05, norm_ones=False), f16)
    toks = np.random.default_rng(4).integers(0, 4500, 6)

    def steps():
        c = gm.make_caches()
        logits = [gm.forward(toks[i:i + 1], i, c) for i in range(4)]
        ids, _, _ = gm.generate_greedy(toks, 6, gm.make_caches())
        return np.stack(logits), np.asarray(ids)

    got = steps()
    with options(ctx, GEMV_BURST="0"):
        want = steps()
    assert np.isfinite(want[0]).all()
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    gm.free()
