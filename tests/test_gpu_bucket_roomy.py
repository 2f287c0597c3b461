"""The largest shape is kept for a few steps after a bucket overflowed a smaller one, no longer than
the second merge is worth."""
import numpy as np
import pytest

from test_gpu_bucket_shapes import _chain_vector
from test_gpu_parity import device_model

pytestmark = pytest.mark.gpu


def test_shape_after_an_overflow(gpu):
    M = N = 20
    rng = np.random.default_rng(4)
    small, _ = _chain_vector(M, N, 250, rng)
    keys, vals = _chain_vector(M, N, 8480, rng)     # 16,960 items: 16 buckets of 1060 on average
    h = device_model(gpu, "real", M, N, 0.0, 1.0)
    e = gpu._native.Engine(h.descriptor(), gpu.IsDynamicSemistochastic().descriptor(), 5, 1 << 18, 1 << 18)
    e.set_timing(True)
    e.upload(small, np.full(250, 1.5))              # the second step has five times the first's attempts
    e.step(1, 4000.0, 1e-3)
    e.step(2, 0.0, 1e-3)
    assert set(e.kernel_times()) & {"bucket_retry", "bucket_fallback"} == {"bucket_retry"}
    assert e.last_cut() == (0, 5)
    cuts = []
    for s in range(3, 16):
        e.upload(keys, vals)
        e.step(s, 0.0, 1e-3)
        cuts.append(e.last_cut()[1])
    e.close()
    print(cuts, flush=True)
    assert cuts[:8] == [5] * 8 and cuts[8:] == [3] * 5
