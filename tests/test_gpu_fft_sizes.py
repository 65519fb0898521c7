"""Binary32 Poisson solve and spectral gradient over the 3 * 2^a mesh sizes (and
the smallest 2^a ones) against the oracle.  The bounds are those of the other
sizes: a two-level transform rounds each value log2(N) times or less per
dimension, 2e-6 = 17 binary32 roundings RMS, and the force meshes carry the
1e-4 of the binary32 force."""
import numpy as np
import pytest

from conftest import clumpy_particles

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda:0")


@pytest.mark.parametrize("N", [8, 12, 24, 32, 96, 384])
def test_potential_fp32_sizes(gpu, oracle_mod, N):
    from hyowon_amd import PMSolver
    L = 2.0 * N
    src = np.random.default_rng(N + 1).standard_normal((N, N, N)).astype(np.float32)
    phi = PMSolver(L, N, precision="fp32", max_particles=1).potential(_dev(src.astype(np.float64)))
    ref = oracle_mod.irfftn(oracle_mod.green_apply(oracle_mod.rfftn(src.astype(np.float64)), L))
    err = np.sqrt(np.mean((phi.cpu().numpy() - ref) ** 2) / np.mean(ref ** 2))
    assert err < 2e-6, err


@pytest.mark.parametrize("prec,N,tol", [("fp32", 24, 1e-4), ("fp32", 96, 1e-4), ("fp32", 192, 1e-4),
                                        ("fp64", 48, 1e-10), ("fp64", 192, 1e-10)])
def test_force_meshes_sizes(gpu, oracle_mod, prec, N, tol):
    from hyowon_amd import PMSolver
    n, L = 20000, 1.25 * N
    pos = clumpy_particles(n, L, 3, sigma=L / 40)
    rs = 1.7 * L / 40
    s = PMSolver(L, N, precision=prec, max_particles=n, method="treepm_long_range", split_scale=rs)
    got = s.force_meshes(s.density(*(_dev(p) for p in pos), None, 1.3))
    *_, ref = oracle_mod.pm_force_treepm(*pos, L, N, rs, uniform_mass=1.3, meshes=True)
    for g, r in zip(got, ref):
        assert np.abs(g.double().cpu().numpy() - r).max() < tol * np.abs(r).max()
