"""The vector-Jacobian product of one fused step against automatic differentiation of the
same force in plain binary64 torch on the host: meshes of 2^a and 3 * 2^a, and particle
sets whose signed deposits take the binary64 deposit's second launch (dense tiles,
long lists, a cell above the LDS key array).

Bounds, relative to the largest component: binary64 1e-10 (sums of up to 3e4 terms and
transforms, at 1e-16 each, with a factor 1e2 for cancellation in the differences);
binary32 2e-4 (the binary32 force's own bound is 1e-4, and the product holds two)."""
import numpy as np
import pytest

from conftest import clumpy_particles

pytestmark = pytest.mark.gpu


def _reference(pos, u, L, N, mass, ksum):
    """ksum * d(sum_p u_p . g(x_p)) / dx, g the centred-gradient CIC force."""
    import math

    import torch
    from hyowon_amd import gravitational_constant
    dx = L / N
    x = [torch.tensor(p, requires_grad=True) for p in pos]
    s = [(v / dx) for v in x]
    base = [t.detach().floor().clamp(max=N - 1) for t in s]
    f = [t - b for t, b in zip(s, base)]
    i = [b.long() for b in base]
    corners = []
    for o in range(8):
        d = [(o >> 2) & 1, (o >> 1) & 1, o & 1]
        w = 1.0
        for a in range(3):
            w = w * (f[a] if d[a] else 1.0 - f[a])
        cell = [(i[a] + d[a]) % N for a in range(3)]
        corners.append((w, (cell[0] * N + cell[1]) * N + cell[2]))
    rho = torch.zeros(N ** 3, dtype=torch.float64)
    for w, c in corners:
        rho = rho.index_add(0, c, w * mass)
    src = (rho - rho.mean()).view(N, N, N) / dx ** 3
    h = math.pi * torch.fft.fftfreq(N, dtype=torch.float64)
    lap = -4.0 / dx ** 2 * torch.sin(h) ** 2
    lap3 = lap.view(-1, 1, 1) + lap.view(1, -1, 1) + lap[: N // 2 + 1].view(1, 1, -1)
    lap3[0, 0, 0] = 1.0
    green = 4.0 * math.pi * gravitational_constant() / lap3
    green[0, 0, 0] = 0.0
    phi = torch.fft.irfftn(torch.fft.rfftn(src) * green, s=(N, N, N))
    total = 0.0
    for a in range(3):
        grad = (-(torch.roll(phi, -1, a) - torch.roll(phi, 1, a)) / (2.0 * dx)).reshape(-1)
        force = sum(w * grad[c] for w, c in corners)
        total = total + (torch.tensor(u[a]) * force).sum()
    (ksum * total).backward()
    return np.stack([t.grad.numpy() for t in x])


def _hot(n, L, N, seed):
    """A background, a ball that makes lists of tens, and one cell of 6000."""
    rng = np.random.default_rng(seed)
    dx = L / N
    pos = rng.uniform(0.0, L, (3, n))
    pos[:, :3000] = np.mod(0.3 * L + rng.normal(0.0, 0.6 * dx, (3, 3000)), L)
    pos[:, 3000:9000] = (N // 2 + 0.5 + rng.uniform(-0.2, 0.2, (3, 6000))) * dx
    return pos[:, rng.permutation(n)]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-10), ("fp32", 2e-4)])
@pytest.mark.parametrize("N,n,kind", [(24, 5000, "clumpy"), (32, 30000, "uniform"), (48, 20000, "clumpy"),
                                      (96, 40000, "clumpy"), (32, 20000, "hot"), (12, 20000, "hot")])
def test_step_vjp(gpu, N, n, kind, prec, tol):
    import torch

    import hyowon_amd as H
    from hyowon_amd._lib import HY_HAS_NEXT, HY_HAS_PREV, check, lib
    from hyowon_amd.pm import _ptr
    L, mass, kp, kn, dn = 1.25 * N, 0.8, 0.02, 0.03, 0.05
    pos = {"clumpy": lambda: clumpy_particles(n, L, 5), "hot": lambda: _hot(n, L, N, 6),
           "uniform": lambda: np.random.default_rng(7).uniform(0.0, L, (3, n))}[kind]()
    rng = np.random.default_rng(N)
    lx0, lp0 = rng.normal(0, 1.0, (3, n)), rng.normal(0, 1.0, (3, n))
    u = lp0 + dn * lx0
    ref = lx0 + _reference(pos, u, L, N, mass, kp + kn)
    s = H.PMSolver(L, N, precision=prec, max_particles=n)
    dev = [torch.as_tensor(np.ascontiguousarray(a), device=gpu) for a in (*pos, *lx0, *lp0)]
    check(lib().hy_pm_kdk_vjp(s.handle, n, *(_ptr(t) for t in dev[:3]), mass, *(_ptr(t) for t in dev[3:]),
                              kp, kn, dn, HY_HAS_PREV | HY_HAS_NEXT))
    got = np.stack([t.cpu().numpy() for t in dev[3:6]])
    assert np.array_equal(np.stack([t.cpu().numpy() for t in dev[6:]]), u)
    err = np.abs((got - lx0) - (ref - lx0)).max() / np.abs(ref - lx0).max()
    assert err < tol, err
