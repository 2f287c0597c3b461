"""Ranked-basis products at the edges of their kernels: two rows, fewer rows than a workgroup
and more, the shortest and longest rings, every number of right-hand sides.

Bars as for the products at ordinary sizes: H.v within 1e-12 relative of the oracle, the adjoint
within 1e-12 of explicit matrices, Lanczos within 1e-9 of a dense eigenvalue.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

# (M, N): dimensions 2, 64 and 63 (64-bit addresses), 253 and 276 (below and above a workgroup of
# 256 rows), 495, 820 (a ring of 40 modes) and 2016 (64-bit addresses)
SPACES = [(2, 1), (2, 63), (63, 1), (22, 2), (23, 2), (5, 8), (40, 2), (63, 2)]


@pytest.mark.parametrize("M,N", SPACES)
@pytest.mark.parametrize("R", range(1, 9))
def test_apply_and_pullback(gpu, M, N, R):
    addr = gpu.near_uniform(N, M)
    us, ts = np.linspace(0.5, 6.0, R), np.linspace(1.0, 0.4, R)
    d = gpu.DenseHamiltonians([gpu.HubbardReal1D(addr, u=u, t=t) for u, t in zip(us, ts)])
    basis = d.basis()
    assert np.array_equal(basis, O.build_basis(M, N))
    rng = np.random.default_rng(1000 * M + 10 * N + R)
    v, ybar = rng.normal(size=(2, d.dim, R))
    a, b = np.linspace(-1.0, 1.0, R), np.linspace(0.7, -0.2, R)
    w = d.apply(a, b, v)
    wo = O.apply_affine([O.real1d(M, N, u, t) for u, t in zip(us, ts)], basis, a, b, v)
    np.testing.assert_allclose(w, wo, rtol=1e-12, atol=1e-12 * np.abs(wo).max())
    vbar, ubar, tbar = d.pullback(a, b, v, ybar)
    Dm = O.sparse_hamiltonian(O.real1d(M, N, 1.0, 0.0), basis)
    Km = O.sparse_hamiltonian(O.real1d(M, N, 0.0, 1.0), basis)
    for i in range(R):
        H = us[i] * Dm + ts[i] * Km
        ref = a[i] * ybar[:, i] + b[i] * (H.T @ ybar[:, i])
        np.testing.assert_allclose(vbar[:, i], ref, rtol=1e-12, atol=1e-12 * np.abs(ref).max())
        # sums over the rows: bounded against the sum of their magnitudes
        for got, G in ((ubar[i], Dm), (tbar[i], Km)):
            mag = np.abs(ybar[:, i]) @ (abs(G) @ np.abs(v[:, i]))
            assert abs(got - b[i] * ybar[:, i] @ (G @ v[:, i])) <= 1e-12 * abs(b[i]) * mag + 1e-300


@pytest.mark.parametrize("M,N", [(2, 1), (2, 63), (23, 2), (5, 8)])
@pytest.mark.parametrize("R", [1, 3, 8])
def test_ground_states(gpu, M, N, R):
    addr = gpu.near_uniform(N, M)
    us = np.linspace(0.5, 6.0, R)
    d = gpu.DenseHamiltonians([gpu.HubbardReal1D(addr, u=u) for u in us])
    basis = d.basis()
    got, _ = d.ground_state()
    for i, u in enumerate(us):
        H = O.sparse_hamiltonian(O.real1d(M, N, u, 1.0), basis).toarray()
        assert got[i] == pytest.approx(np.linalg.eigvalsh(H)[0], rel=1e-9, abs=1e-9)
