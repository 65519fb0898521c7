"""The binary64 deposit where its plan of a dense tile does not fit the job list: the tile is
cut evenly, jobs above the LDS list their records in the scratch and halve
their boxes on the stack, and jobs that find the scratch full go through the tile's
records each time.  Bit for bit against the oracle; tile edges of 16, 12 and 8."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (mesh, uniform particles, particles in a ball, ball radius in cells)
DENSE = [
    (16, 60000, 0, 0.0),       # one tile, over 100 leaves against 64 list entries
    (24, 300000, 0, 0.0),      # edge 12, eight tiles: the list's 512 entries run out part way
    (8, 30000, 0, 0.0),        # edge 8, one tile that is its own neighbour
    (8, 70000, 0, 0.0),        # 64 jobs list 3.4 n records; the scratch holds 2 n + 65536
    (8, 60000, 20000, 0.2),    # and cells above the LDS key array
    (16, 60000, 30000, 0.3),
]


@pytest.mark.parametrize("N,nu,nb,radius", DENSE)
@pytest.mark.parametrize("explicit", [False, True])
def test_density_without_a_plan_bit_exact(gpu, oracle_mod, N, nu, nb, radius, explicit):
    import torch

    import hyowon_amd as H
    rng = np.random.default_rng(N + nu + nb)
    L = 1.0 * N
    pos = rng.uniform(0.0, L, (3, nu))
    if nb:
        centre = np.array([N // 2, 0.0, N // 2 + 0.4]).reshape(3, 1)
        pos = np.concatenate([pos, np.mod(centre + rng.normal(0.0, radius, (3, nb)), L)], axis=1)
    pos = np.ascontiguousarray(pos[:, rng.permutation(pos.shape[1])])
    n = pos.shape[1]
    masses = rng.uniform(0.5, 2.0, n) if explicit else None
    s = H.PMSolver(L, N, precision="fp64", max_particles=n)
    got = s.density(*(torch.as_tensor(p, device=gpu) for p in pos),
                    torch.as_tensor(masses, device=gpu) if explicit else None, 0.0 if explicit else 0.75)
    if explicit:
        dep = oracle_mod.deposit(*pos, L, N, masses=masses)
        total = float(oracle_mod.lib().or_exact_sum(masses.ctypes.data_as(oracle_mod._pd), n))
    else:
        dep, total = oracle_mod.deposit(*pos, L, N, uniform_mass=0.75), 0.75 * n
    assert np.array_equal(got.cpu().numpy(), oracle_mod.density_contrast(dep, L, N, total))
