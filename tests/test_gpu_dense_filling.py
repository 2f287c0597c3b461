"""Ranked-basis products on both sides of the filling where they change from walking the occupied
modes to passing over all bonds, and what few bosons on many modes may cost.

Bar as for the products at other sizes: within 1e-12 relative of the oracle.
"""
import time

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


# up to four right-hand sides the line lies at 2 N = M, above that at 3 N = 2 M; 300 rows or more
# leave a ragged last workgroup
@pytest.mark.parametrize("M,N", [(3, 1), (2, 1), (9, 4), (8, 4), (9, 6), (10, 7), (13, 6), (64, 1)])
@pytest.mark.parametrize("R", [1, 4, 5, 8])
def test_products_at_the_line(gpu, M, N, R):
    addr = gpu.near_uniform(N, M)
    us, ts = np.linspace(0.5, 6.0, R), np.linspace(1.0, 0.4, R)
    d = gpu.DenseHamiltonians([gpu.HubbardReal1D(addr, u=u, t=t) for u, t in zip(us, ts)])
    basis = d.basis()
    rng = np.random.default_rng(1000 * M + 10 * N + R)
    v, ybar = rng.normal(size=(2, d.dim, R))
    a, b = np.linspace(-1.0, 1.0, R), np.linspace(0.7, -0.2, R)
    hs = [O.real1d(M, N, u, t) for u, t in zip(us, ts)]
    w = d.apply(a, b, v)
    wo = O.apply_affine(hs, basis, a, b, v)
    np.testing.assert_allclose(w, wo, rtol=1e-12, atol=1e-12 * np.abs(wo).max())
    vbar, _, _ = d.pullback(a, b, v, ybar)
    vo = O.apply_affine(hs, basis, a, b, ybar)   # H is symmetric
    np.testing.assert_allclose(vbar, vo, rtol=1e-12, atol=1e-12 * np.abs(vo).max())


def test_few_bosons_on_many_modes_cost_their_hops(gpu):
    """At most 8 hops a row (4 bosons on 60 modes) and up to 16 (8 on 16) at similar dimensions:
    a pass over all bonds made the first 2.7 times as slow as the second."""
    ms = {}
    for M, N in ((60, 4), (16, 8)):
        d = gpu.DenseHamiltonians([gpu.HubbardReal1D(gpu.near_uniform(N, M), u=u) for u in (1.0, 2.0, 3.0, 4.0)])
        v0 = d.unit_vector(gpu.near_uniform(N, M))
        t = []
        for _ in range(6):
            t0 = time.perf_counter()
            d.projector_energy(200, 1e-3, 0.0, v0)
            t.append(time.perf_counter() - t0)
        ms[M] = 1e3 * sorted(t)[2]
        d.close()
    print(ms, flush=True)
    assert ms[60] < 1.6 * ms[16]
