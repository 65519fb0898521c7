"""The binary64 deposit's work splits, bit for bit against the oracle: tiles
whose records exceed the workgroup's LDS (jobs planned from their record counts;
where no plan fits: test_gpu_deposit_fallback.py), long cell lists (one wave each),
single cells hotter than the LDS list and than the LDS key array, tiles that are
not 16 cells wide, explicit masses."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ball(n, L, centre, radius, seed):
    rng = np.random.default_rng(seed)
    return np.mod(np.asarray(centre).reshape(3, 1) + rng.normal(0.0, radius, (3, n)), L)


# (mesh, L, uniform background, particles in a ball, ball radius in cells)
SPLITS = [
    (32, 32.0, 8192, 0, 0.0),        # 1/4 per cell: two boxes per tile
    (48, 60.0, 110592, 0, 0.0),      # one per cell, cell size not a power of two
    (24, 24.0, 6000, 600, 0.2),      # tile edge 12, lists longer than one thread sorts
    (8, 8.0, 500, 5000, 1.0),        # tile edge 8, periodic neighbours are the tile itself
    (32, 32.0, 4000, 3000, 0.4),     # cells above the LDS list
    (32, 40.0, 4000, 30000, 0.3),    # cells above the LDS key array
    # one cell's neighbourhood, 1124 and 1126 records with the periodic duplicates: planned
    # (record counts at the kernels' capacities: test_gpu_deposit_capacity.py)
    (16, 16.0, 1, 767, 0.05),
    (16, 16.0, 1, 768, 0.05),
]


@pytest.mark.parametrize("N,L,nu,nb,radius", SPLITS)
@pytest.mark.parametrize("explicit", [False, True])
def test_density_fp64_dense_tiles_bit_exact(gpu, oracle_mod, N, L, nu, nb, radius, explicit):
    import torch

    import hyowon_amd as H
    rng = np.random.default_rng(N + nu + nb)
    dx = L / N
    pos = rng.uniform(0.0, L, (3, nu))
    if nb:
        # across a tile corner and the periodic boundary (cell 0 along y)
        pos = np.concatenate([pos, _ball(nb, L, ((N // 2) * dx, 0.0, (N // 2 + 0.4) * dx), radius * dx, 5)], axis=1)
    pos = pos[:, rng.permutation(pos.shape[1])]
    n = pos.shape[1]
    masses = rng.uniform(0.5, 2.0, n) if explicit else None
    m = 0.75
    s = H.PMSolver(L, N, precision="fp64", max_particles=n)
    t = [torch.as_tensor(np.ascontiguousarray(p), device=gpu) for p in pos]
    mt = torch.as_tensor(masses, device=gpu) if explicit else None
    mesh = s.density(*t, mt, 0.0 if explicit else m).cpu().numpy()
    if explicit:
        dep = oracle_mod.deposit(pos[0], pos[1], pos[2], L, N, masses=masses)
        total = float(oracle_mod.lib().or_exact_sum(masses.ctypes.data_as(oracle_mod._pd), n))
    else:
        dep = oracle_mod.deposit(pos[0], pos[1], pos[2], L, N, uniform_mass=m)
        total = m * n
    ref = oracle_mod.density_contrast(dep, L, N, total)
    assert np.array_equal(mesh, ref), np.abs(mesh - ref).max()
