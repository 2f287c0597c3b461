"""The largest shape is kept for a few steps after a bucket overflowed a smaller one, no longer than
the second merge is worth."""
import numpy as np
import pytest

from test_gpu_bucket_shapes import _chain_vector
from test_gpu_parity import device_model

pytestmark = pytest.mark.gpu


def test_shape_after_an_overflow(gpu):
    """Sixteen steps after the first overflow; 64 after one that comes soon after those; sixteen
    after one that does not."""
    M = N = 20
    rng = np.random.default_rng(4)
    small, _ = _chain_vector(M, N, 250, rng)
    keys, vals = _chain_vector(M, N, 8480, rng)     # 16,960 items: 16 buckets of 1060 on average
    h = device_model(gpu, "real", M, N, 0.0, 1.0)
    e = gpu._native.Engine(h.descriptor(), gpu.IsDynamicSemistochastic().descriptor(), 5, 1 << 18, 1 << 18)
    e.set_timing(True)
    step = 0

    def overflow():
        nonlocal step
        e.upload(small, np.full(250, 1.2))          # two small steps, the second sized by the first
        e.step(step + 1, 0.0, 1e-3)
        e.upload(small, np.full(250, 1.2))
        e.step(step + 2, 0.0, 1e-3)
        e.upload(small, np.full(250, 6.5))          # five times their attempts
        e.step(step + 3, 0.0, 1e-3)
        step += 3
        return e.kernel_times().get("bucket_retry", (0, 0))[1], e.last_cut()

    def shapes(n):
        nonlocal step
        out = []
        for _ in range(n):
            step += 1
            e.upload(keys, vals)
            e.step(step, 0.0, 1e-3)
            out.append(e.last_cut()[1])
        return out

    assert overflow() == (1, (0, 5))
    assert shapes(21) == [5] * 16 + [3] * 5
    assert overflow() == (2, (0, 5))
    assert shapes(69) == [5] * 64 + [3] * 5
    assert shapes(256) == [3] * 256
    assert overflow() == (3, (0, 5))
    assert shapes(21) == [5] * 16 + [3] * 5
    assert "bucket_fallback" not in e.kernel_times()
    e.close()
