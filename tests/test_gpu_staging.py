"""Small transfers between host and device go through page-locked memory and a copy kernel of 16-byte pieces; larger ones do not."""
import numpy as np
import pytest

import rllama_amd
from common import Shape, make_gpu, synth_weights
from rllama_amd import Tensor

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx():
    """A context of its own: what these tensors leave in the pool of freed buffers goes with it."""
    c = rllama_amd.Context(0)
    yield c
    c.close()


# bytes: less than a piece, pieces and every kind of rest, more than the kernel has threads, the staging's 1 MiB and one element around it
@pytest.mark.parametrize("cols", [1, 3, 7, 8, 9, 15, 16, 17, 2047, 2049, 32000, 65536 * 8 - 1, 65536 * 8, 65536 * 8 + 1])
@pytest.mark.parametrize("dtype", [np.uint16, np.float32])
def test_download_returns_what_was_uploaded(ctx, cols, dtype):
    rng = np.random.default_rng(cols)
    if dtype == np.float32:
        cols = (cols + 1) // 2
    for _ in range(3):  # the staging is reused
        a = rng.integers(0, 1 << 15, (1, cols)).astype(dtype)
        assert np.array_equal(Tensor.from_numpy(ctx, a).to_numpy().reshape(a.shape).view(dtype), a)


def test_prompts_behind_calls_that_read_ids_only(ctx):
    """The greedy calls upload a prompt and read ids: the next call's prompt must not overwrite ids that are still queued, nor the other way round."""
    shape = Shape(dim=256, n_layers=2, n_heads=4, ffn_hidden=512, vocab_size=300, max_seq_len=64)
    gm = make_gpu(ctx, shape, synth_weights(shape, seed=5, std=0.05, norm_ones=False), True)
    rng = np.random.default_rng(6)
    prompts = [rng.integers(0, 300, n) for n in (2, 40, 7, 33)]
    want = [gm.forward(p, 0, gm.make_caches()) for p in prompts]
    picks = [int(gm.forward_greedy(p, 0, gm.make_caches())) for p in prompts]
    for p, w, pick in zip(prompts, want, picks):
        ids, _, _ = gm.generate_greedy(p, 5, gm.make_caches())
        assert int(ids[0]) == pick
        for q, w2 in zip(prompts, want):
            assert np.array_equal(gm.forward(q, 0, gm.make_caches()), w2)
            assert int(gm.forward_greedy(p, 0, gm.make_caches())) == pick
    gm.free()
