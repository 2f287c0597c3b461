"""Where vectors change from the host's sort to the device's between address order and stored-key
order: 1024 entries and 56 for every key bit."""
import numpy as np
import pytest

from test_gpu_parity import device_model
from test_gpu_reorder import _wide

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(12, 10), (20, 20), (33, 33), (64, 64)])   # 21, 39, 65, 127 bits
@pytest.mark.parametrize("below", [1, 0])
def test_route_and_order_at_the_line(gpu, M, N, below):
    bits = M + N - 1
    n = 1024 + 56 * bits - below
    rng = np.random.default_rng(bits)
    keys, m = _wide(M, N, 3 * n, rng)
    keys = keys[np.sort(rng.permutation(m)[:n])]
    assert len(keys) == n
    if bits <= 64:
        keys = np.ascontiguousarray(keys[:, 0])
    vals = rng.normal(size=n)
    h = device_model(gpu, "real", M, N, 4.0, 1.0)
    e = gpu._native.Engine(h.descriptor(), gpu.IsDeterministic().descriptor(), 3, 4 * n, 4 * n)
    e.set_timing(True)
    scatters = []
    for go in (lambda: e.upload(keys, vals), e.download):
        got = go()
        gpu._native.overlaps(e, e)                       # ends the timing of what ran before it
        scatters.append(e.kernel_times().get("radix_scatter", (0, 0))[1])
    e.close()
    if below:
        assert scatters == [0, 0]
    else:
        assert 0 < scatters[0] < scatters[1]
    assert np.array_equal(got[0], keys) and np.array_equal(got[1], vals)
