"""Buffers of freed op-level tensors are used again: results stay those of fresh tensors, new tensors are zero, padded rows survive."""
import numpy as np
import pytest

from rllama_amd import Tensor, TensorDType

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


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (2048, 1024), (2049, 1024)])  # the last is over the size that is kept
def test_upload_and_download_of_reused_buffers(ctx, rows, cols):
    rng = np.random.default_rng(rows)
    for _ in range(4):
        x = rng.standard_normal((rows, cols)).astype(np.float32)
        t = Tensor.from_numpy(ctx, x)
        assert np.array_equal(t.to_numpy(), x)
        t.free()
