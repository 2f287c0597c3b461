"""A bucket that overflows a small shape is merged again in the largest; one that overflows that too
goes along the merge path.  Steps sized by the one before meet both when the walkers multiply."""
import numpy as np
import pytest

from test_gpu_bucket_shapes import _chain_vector
from test_gpu_parity import device_model

pytestmark = pytest.mark.gpu


# 250 entries of 1.01 .. 1.99 whose values the first step multiplies by 1 + 1e-3 shift: the second
# has about 250 x that many attempts in one bucket planned for 500 items in the smallest shape (1536)
@pytest.mark.parametrize("shift,label", [(1.0, None), (4000.0, "bucket_retry"), (12_000.0, "bucket_fallback")])
def test_overflow_of_a_shape(gpu, shift, label):
    M = N = 20
    rng = np.random.default_rng(3)
    keys, vals = _chain_vector(M, N, 250, rng)
    h = device_model(gpu, "real", M, N, 0.0, 1.0)
    out = []
    for mode in (2, 1):
        e = gpu._native.Engine(h.descriptor(), gpu.IsDynamicSemistochastic().descriptor(), 5, 1 << 18, 1 << 18)
        e.set_radix_mode(mode)
        e.set_timing(True)
        e.upload(keys, vals)
        st = [e.step(1, shift, 1e-3), e.step(2, 0.0, 1e-3), e.step(3, 0.0, 1e-3)]
        out.append((e.download(), [(x.len, x.len_before, x.spawn_attempts) for x in st], set(e.kernel_times())))
        print(f"shift={shift} mode={mode} {out[-1][1]}", flush=True)
        e.close()
    met = out[0][2] & {"bucket_retry", "bucket_fallback"}
    assert (label in met) if label else not met
    assert label != "bucket_retry" or met == {"bucket_retry"}
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0][0], out[1][0][0])
    assert np.array_equal(out[0][0][1].view(np.uint64), out[1][0][1].view(np.uint64))
