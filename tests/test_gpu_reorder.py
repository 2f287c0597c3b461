"""Vectors between address order and stored-key order: the device's sort against the host's
(an engine whose spawn buffers cannot hold the vector takes the host's)."""
import numpy as np
import pytest

from test_gpu_parity import device_model

pytestmark = pytest.mark.gpu


def _wide(M, N, n, rng):
    occ = rng.multinomial(N, np.full(M, 1.0 / M), size=n)
    out = set()
    for row in occ.tolist():
        x, at = 0, 0
        for k in row:
            x |= ((1 << k) - 1) << at
            at += k + 1
        out.add(x)
    keys = sorted(out)
    return np.array([[k & (2 ** 64 - 1), k >> 64] for k in keys], dtype=np.uint64), len(keys)


@pytest.mark.parametrize("M,N", [(16, 16), (32, 33), (33, 33), (50, 50), (64, 65)])   # 31, 64, 65, 99, 128 bits
@pytest.mark.parametrize("n", [1023, 1024, 1025, 6145])
@pytest.mark.parametrize("style", ["integer", "exact"])
def test_device_order_equals_host_order(gpu, M, N, n, style):
    rng = np.random.default_rng(M * n)
    keys, m = _wide(M, N, n, rng)
    vals = rng.integers(1, 50, m) if style == "integer" else rng.normal(size=m)
    vals[5] = 0                                     # zero values are dropped
    st = gpu.IsStochasticInteger() if style == "integer" else gpu.IsDeterministic()
    h = device_model(gpu, "real", M, N, 4.0, 1.0)
    kw = 2 if M + N > 65 else 1
    keys = keys if kw == 2 else np.ascontiguousarray(keys[:, 0])
    want_k, want_v = np.delete(keys, 5, axis=0), np.delete(vals, 5)
    for room in (4 * m, 16):                        # the device's sort, the host's
        e = gpu._native.Engine(h.descriptor(), st.descriptor(), 3, 4 * m, room)
        e.upload(keys, vals)
        k, v = e.download()
        e.close()
        assert np.array_equal(k, want_k) and np.array_equal(v, want_v)


def test_device_order_equals_host_order_after_a_step(gpu):
    """A stored order written by one route is read back by the other."""
    M = N = 50
    rng = np.random.default_rng(9)
    keys, m = _wide(M, N, 3000, rng)
    vals = rng.uniform(1.0, 3.0, m)
    h = device_model(gpu, "real", M, N, 6.0, 1.0)
    out = []
    for room in (16, 1 << 16):
        e = gpu._native.Engine(h.descriptor(), gpu.IsDynamicSemistochastic().descriptor(), 3, 1 << 16, room)
        e.upload(keys, vals)
        e.reserve(1 << 16, 1 << 16)
        e.step(1, -1.0, 1e-3)
        out.append(e.download())
        e.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
