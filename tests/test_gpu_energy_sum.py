"""The potential-energy sum at the edges of its 4096-particle blocks and the
2048-term pieces they are added in, bit for bit against the oracle's ordered
compensated sum, with terms that cancel and differ widely in size."""
import numpy as np
import pytest

from conftest import clumpy_particles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 2047, 2048, 2049, 4095, 4096, 4097, 10240, 70001])
def test_energy_sum_edges(gpu, oracle_mod, n):
    import hyowon_amd as H
    import torch
    N, L = 32, 40.0
    rng = np.random.default_rng(n)
    pos = clumpy_particles(n, L, n)
    masses = 10.0 ** rng.uniform(-12.0, 0.0, n)
    x, y, z, m = (torch.as_tensor(np.ascontiguousarray(v), device=gpu) for v in (*pos, masses))
    s = H.PMSolver(L, N, precision="fp64", max_particles=n)
    phi = s.potential(s.density(x, y, z, m)).cpu().numpy()
    acc = [torch.zeros(n, dtype=torch.float64, device=gpu) for _ in range(3)]
    d = s.compute_forces(x, y, z, m, None, *acc, collect_potential_energy=True)
    assert d.potential_energy_comoving == oracle_mod.potential_energy(phi, *pos, L, masses=masses)
