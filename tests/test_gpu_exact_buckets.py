"""Exact steps: below 4096 records they take the merge path, above it the bucket merge in its largest
shape; the vector is the same bit for bit."""
import numpy as np
import pytest

from test_gpu_bucket_shapes import _chain_vector
from test_gpu_parity import device_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 40, 160, 400, 3000])
def test_exact_steps_take_large_buckets(gpu, n):
    M = N = 20
    rng = np.random.default_rng(n)
    keys, vals = _chain_vector(M, N, n, rng)
    h = device_model(gpu, "real", M, N, 4.0, 1.0)
    out = []
    for mode in (2, 1):
        e = gpu._native.Engine(h.descriptor(), gpu.IsDeterministic().descriptor(), 5, 1 << 20, 1 << 21)
        e.set_radix_mode(mode)
        e.set_timing(True)
        e.upload(keys, vals)
        st = e.step(1, -2.0, 1e-3)
        out.append((st, e.download(), set(e.kernel_times())))
        e.close()
    records = out[0][0].spawn_attempts
    assert ("bucket_merge" in out[0][2]) == (records >= 4096) and "bucket_merge" not in out[1][2]
    assert np.array_equal(out[0][1][0], out[1][1][0])
    assert np.array_equal(out[0][1][1].view(np.uint64), out[1][1][1].view(np.uint64))
    # at most 1e6 terms added in another order
    assert abs(out[0][0].norm - out[1][0].norm) <= 1e-10 * out[1][0].norm
    if records < 4096:
        assert out[0][0].norm == out[1][0].norm
