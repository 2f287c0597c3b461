"""Ground-state energies do not depend on the length of the start vector."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


# |v0|^2 between 3e-306 and 3e307 for 252 rows; <v0|H v0> is some hundred times as large
@pytest.mark.parametrize("scale", [1.0, 1e-154, 1e-100, 1e100, 3e152])
@pytest.mark.parametrize("R", [1, 3])
def test_energies_for_long_and_short_start_vectors(gpu, scale, R):
    M, N = 6, 5
    addr = gpu.near_uniform(N, M)
    us = np.linspace(20.0, 40.0, R)
    d = gpu.DenseHamiltonians([gpu.HubbardReal1D(addr, u=u, t=1.0) for u in us])
    rng = np.random.default_rng(8)
    v0 = scale * rng.uniform(0.5, 1.5, (d.dim, R))
    assert np.all(np.isfinite((v0 * v0).sum(axis=0))) and np.all((v0 * v0).sum(axis=0) > 0)
    got, _ = d.ground_state(v0)
    basis = d.basis()
    for i, u in enumerate(us):
        H = O.sparse_hamiltonian(O.real1d(M, N, u, 1.0), basis).toarray()
        assert got[i] == pytest.approx(np.linalg.eigvalsh(H)[0], rel=1e-9, abs=1e-9)
    with pytest.raises(gpu.RimuError):
        d.ground_state(np.zeros((d.dim, R)))
