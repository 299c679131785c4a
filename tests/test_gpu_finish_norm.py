"""The kernel that adds the pieces of wo and w2 and normalises the row, against the two kernels of their own: same bits."""
import numpy as np
import pytest

from common import Shape, make_gpu, options, synth_weights

pytestmark = pytest.mark.gpu


# rows of the largest width for 256 and 512 threads, one past it, the widest for one piece per thread and one with two; pieces of the kernel for few rows
# (20) and of the tiled ones (200)
@pytest.mark.parametrize("dim,heads", [(1024, 16), (1088, 17), (2048, 16), (2112, 33), (4096, 32), (4160, 65)])
def test_same_bits_as_the_separate_kernels(ctx, dim, heads):
    shape = Shape(dim=dim, n_layers=2, n_heads=heads, ffn_hidden=4096, vocab_size=64, max_seq_len=256)
    gm = make_gpu(ctx, shape, synth_weights(shape, seed=21, std=0.05, norm_ones=False), True)
    toks = np.random.default_rng(22).integers(0, 64, 200)
    for n in (20, 200):
        got = gm.forward(toks[:n], 0, gm.make_caches())
        with options(ctx, FINISH_NORM="0"):
            want = gm.forward(toks[:n], 0, gm.make_caches())
        assert np.isfinite(want).all() and np.array_equal(got, want), n
    gm.free()
