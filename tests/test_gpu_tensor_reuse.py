"""Buffers of freed op-level tensors are used again: results stay those of fresh tensors, new tensors are zero, padded rows survive."""
import numpy as np
import pytest

from rllama_amd import Context, Tensor, TensorDType

pytestmark = pytest.mark.gpu


def test_freed_buffers_come_back_zeroed_and_in_order(ctx):
    rng = np.random.default_rng(3)
    a, b = rng.standard_normal((40, 256)).astype(np.float32), rng.standard_normal((96, 256)).astype(np.float32)
    A, B = Tensor.from_numpy(ctx, a), Tensor.from_numpy(ctx, b)
    first = A.matrix_mul_transposed(B).to_numpy()
    for _ in range(30):  # results dropped while their work may still be queued; the next one takes the same buffer
        A.matrix_mul_transposed(B).silu()
        z = Tensor.zeros(ctx, 40, 96, TensorDType.Float32)
        got = A.matrix_mul_transposed(B)
        assert not z.to_numpy().any()
        assert np.array_equal(got.to_numpy(), first)


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (2048, 1024), (2049, 1024), (8193, 1024)])  # the last is over the size that is kept
def test_upload_and_download_of_reused_buffers(ctx, rows, cols):
    rng = np.random.default_rng(rows)
    for _ in range(4):
        x = rng.standard_normal((rows, cols)).astype(np.float32)
        t = Tensor.from_numpy(ctx, x)
        assert np.array_equal(t.to_numpy(), x)
        t.free()


def test_tensors_of_changing_sizes(ctx):
    """More sizes than the pool holds, in buffers of larger ones: new tensors are zero to their end, contents are their own."""
    rng = np.random.default_rng(5)
    kept = []
    for i in range(400):
        rows = int(rng.integers(1, 700))
        z = Tensor.zeros(ctx, rows, 4100, TensorDType.Float32)
        x = rng.standard_normal((rows, 11)).astype(np.float32)
        kept.append((x, Tensor.from_numpy(ctx, x)))
        if i % 10 == 0:
            assert not z.to_numpy().any()
            for want, t in kept:
                assert np.array_equal(t.to_numpy(), want)
            kept = kept[-3:]


def test_buffers_that_another_context_uses_are_not_handed_out(ctx):
    """A tensor freed while an operation of another context (another stream) reads it: a new tensor of its size must not get the buffer."""
    rng = np.random.default_rng(4)
    other = Context(0)
    try:
        x = Tensor.from_numpy(other, rng.standard_normal((512, 1024)).astype(np.float32))
        w = rng.standard_normal((2048, 1024)).astype(np.float32)
        junk = np.full_like(w, 7.0)
        want = x.matrix_mul_transposed(Tensor.from_numpy(other, w)).to_numpy()
        for _ in range(20):
            W = Tensor.from_numpy(ctx, w)
            for _ in range(4):  # work of the other context that is still queued when the tensor is freed
                got = x.matrix_mul_transposed(W)
            W.free()
            J = Tensor.from_numpy(ctx, junk)
            assert np.array_equal(got.to_numpy(), want)
            assert np.array_equal(J.to_numpy(), junk)
    finally:
        other.close()
