"""Steps whose statistics, scans and compactions fit one workgroup against those that do not:
the sizes around the limits (1024 tiles of each kind), through the oracle's integer steps."""
import numpy as np
import pytest

import oracle as O
from test_gpu_bucket_shapes import _chain_vector
from test_gpu_parity import device_model, oracle_model

pytestmark = pytest.mark.gpu


# spawn tiles hold 1024 attempts: 1024 and 1025 of them, and one; entries of one walker or so
@pytest.mark.parametrize("attempts", [1, 1023, 1024 * 1024 - 1, 1024 * 1024, 1024 * 1024 + 1])
def test_spawn_tiles_around_the_limits(gpu, attempts):
    M = N = 16
    rng = np.random.default_rng(attempts)
    n = min(attempts, 40_000)
    keys, _ = _chain_vector(M, N, n, rng)
    vals = np.full(n, attempts // n, dtype=np.int64)
    vals[0] += attempts - int(vals.sum())
    vals *= rng.choice([-1, 1], n)
    h = device_model(gpu, "real", M, N, 6.0, 1.0)
    e = gpu._native.Engine(h.descriptor(), gpu.IsStochasticInteger().descriptor(), 11, 1 << 21, 1 << 21)
    e.upload(keys, vals)
    pk = keys[:200]
    e.set_projector(pk, np.arange(1.0, len(pk) + 1), pk[:1], np.ones(1))
    om = oracle_model("real", M, N, 6.0, 1.0)
    k, v = keys, vals
    for step in (1, 2, 3):                          # the first step reads its counts back
        st = e.step(step, -1.0, 1e-3)
        k, v, ost = O.step(om, O.style("integer"), k, v, seed=11, step=step, shift=-1.0, dtau=1e-3, order=1)
        gk, gv = e.download()
        assert np.array_equal(gk, k) and np.array_equal(gv, v)
        assert (st.spawn_attempts, st.norm, st.len) == (ost["attempts"], ost["norm"], len(k))
        d = dict(zip(k.tolist(), v.tolist()))
        assert st.vproj == sum((i + 1.0) * d.get(x, 0) for i, x in enumerate(pk.tolist()))
    e.close()
