"""Overlaps at the edges of their tiles and of the left vector's index, against the oracle."""
import numpy as np
import pytest

import oracle as O
from test_gpu_bucket_shapes import _chain_vector
from test_gpu_parity import device_model, oracle_model

pytestmark = pytest.mark.gpu


# the index starts at 4096 left keys; tiles are 512 right entries, a round of the Hamiltonian
# kernel 32 entries per workgroup
@pytest.mark.parametrize("nl", [1, 3, 4, 1023, 4095, 4096, 4097])
@pytest.mark.parametrize("nr", [1, 33, 511, 513, 5000])
def test_overlap_sizes(gpu, nl, nr):
    M = N = 20                                    # 39-bit mixed keys
    rng = np.random.default_rng(nl * 7 + nr)
    pool, vals = _chain_vector(M, N, max(nl, nr) + 100, rng)
    h = device_model(gpu, "real", M, N, 4.0, 1.0)
    st = gpu.IsDeterministic()
    vec = []
    for n in (nl, nr):
        at = np.sort(rng.choice(len(pool), n, replace=False))
        e = gpu._native.Engine(h.descriptor(), st.descriptor(), 1, n + 10, 1 << 16)
        e.upload(pool[at], vals[at])
        vec.append((e, pool[at], vals[at]))
    (a, lk, lv), (b, rk, rv) = vec
    ops = [gpu.G2RealCorrelator(1), h, gpu.DensityMatrixDiagonal(2), h]
    got = gpu.observables.overlap_values(gpu.DeviceDVec(a, h, st), gpu.DeviceDVec(b, h, st), ops)
    a.close()
    b.close()
    om = oracle_model("real", M, N, 4.0, 1.0)
    want = O.overlaps(lk, lv, rk, rv, M, [("g2", 1), ("ham", om), ("density", 2), ("ham", om)])
    scale = np.abs(lv).sum() * np.abs(rv).max() * 10
    np.testing.assert_allclose(got, want, rtol=1e-12, atol=1e-13 * scale)
