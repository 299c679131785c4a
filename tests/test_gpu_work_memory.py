"""How much work memory op-level products and prompts hold on the device."""
import ctypes
import gc

import numpy as np
import pytest

import rllama_amd
from common import SMALL, make_gpu, random_f32_weights
from rllama_amd import Context, Tensor

pytestmark = pytest.mark.gpu
MB = 1 << 20


def _used():
    """Bytes in use on the device, from the HIP runtime that the library has loaded."""
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return total.value - free.value


def _product(c, m, n, k, dtype):
    x = Tensor.from_numpy(c, np.ones((m, k), dtype)), Tensor.from_numpy(c, np.ones((n, k), dtype))
    y = x[0].matrix_mul_transposed(x[1])
    assert (y.to_numpy() == k).all()
    for t in (*x, y):
        t.free()


def test_op_level_products_hold_what_they_need(ctx):
    _product(ctx, 64, 256, 256, np.float16)  # what the process needs once
    c = Context(0)
    try:
        before = _used()
        _product(c, 64, 256, 256, np.float16)
        _product(c, 64, 256, 256, np.float32)
        assert _used() - before < 100 * MB  # 64 for partial sums, the kept buffers, the runtime's granularity
        _product(c, 1200, 1024, 8192, np.float32)  # 60 MB of parts, 16 pieces of 5 MB
        assert 100 * MB < _used() - before < 300 * MB
    finally:
        c.close()


def test_short_f32_prompts_hold_no_more_than_short_f16_ones(ctx):
    gm = make_gpu(ctx, SMALL, random_f32_weights(SMALL, 3), False)
    caches = gm.make_caches()
    gc.collect()
    before = _used()
    gm.forward(np.arange(8), 0, caches)
    assert _used() - before < 100 * MB
    gm.free()
