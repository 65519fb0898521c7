"""The binary64 deposit's first launch at the record counts of a tile where its
kernels end (736 narrow, 1024 wide), bit for bit against the oracle: one record per
base cell, none on a tile's last cells, so a tile's count is its own particles
and no list is long.  The mean over the tiles chooses the kernel."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FULL = [736, 737, 1023, 1024, 1025, 900, 800, 700]          # all eight tiles of 32^3: wide
SPARSE = [735, 736, 737, 1024, 1025]                        # five of the 64 tiles of 64^3: narrow


@pytest.mark.parametrize("N,counts", [(32, FULL), (64, SPARSE)])
@pytest.mark.parametrize("explicit", [False, True])
def test_tile_counts_at_the_capacities(gpu, oracle_mod, N, counts, explicit):
    import torch

    import hyowon_amd as H
    T, L = 16, 1.25 * N
    nT = N // T
    rng = np.random.default_rng(N + explicit)
    pos = []
    for k, m in enumerate(counts):
        t = k * (nT ** 3 // len(counts))
        cells = rng.permutation((T - 1) ** 3)[:m]
        base = np.stack([cells // (T - 1) ** 2, cells // (T - 1) % (T - 1), cells % (T - 1)])
        corner = T * np.array([t // nT ** 2, t // nT % nT, t % nT]).reshape(3, 1)
        pos.append((corner + base + rng.uniform(0.05, 0.95, base.shape)) * (L / N))
    pos = np.concatenate(pos, axis=1)
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


def test_time_does_not_jump_between_the_capacities(gpu):
    """256^3, lattice loads of 0.14 and 0.165 particles per cell (688 and 811 records a
    tile): 18% more particles must not cost what a second pass over them does (1.5)."""
    import torch

    import hyowon_amd as H
    N = 256

    def timed(S):
        g = torch.Generator(device="cuda").manual_seed(S)
        q = (torch.arange(S, device="cuda", dtype=torch.float64) + 0.5) * (N / S)
        pos = [torch.remainder(a.reshape(-1) + 0.5 * torch.randn(S ** 3, device="cuda", dtype=torch.float64, generator=g), N)
               for a in torch.meshgrid(q, q, q, indexing="ij")]
        s = H.PMSolver(float(N), N, precision="fp64", max_particles=S ** 3)
        times = []
        for _ in range(12):
            torch.cuda.synchronize()
            t = time.perf_counter()
            s.density(*pos, None, 1.0)
            times.append(time.perf_counter() - t)
        return sorted(times)[5]

    light, full = timed(133), timed(140)
    assert full < 1.35 * light, (full, light)
