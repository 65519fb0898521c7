"""Forces of a million particles and more, gathered in particle order where the order
keeps to the deposit buckets (near a lattice, sorted) and in record order where it does
not: the bits of the particle-order gather and interpolation either way, and an
in-order call that costs no more than the step of the same particles, which
gathers in particle order."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _positions(order, S, L):
    import torch
    g = torch.Generator(device="cuda").manual_seed(S)
    q = (torch.arange(S, device="cuda", dtype=torch.float64) + 0.5) * (L / S)
    pos = [torch.remainder(a.reshape(-1) + 0.3 * (L / S) * torch.randn(S ** 3, device="cuda", dtype=torch.float64, generator=g), L)
           for a in torch.meshgrid(q, q, q, indexing="ij")]
    if order == "shuffled":
        p = torch.randperm(S ** 3, device="cuda", generator=g)
        pos = [x[p].contiguous() for x in pos]
    return pos


@pytest.mark.parametrize("order", ["lattice", "shuffled"])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N,method,explicit", [(192, "pure_pm", False), (128, "pure_pm", True), (192, "treepm_long_range", False)])
def test_both_orders_give_the_same_bits(gpu, N, method, explicit, prec, order):
    import torch

    import hyowon_amd as H
    S, L = 102, 1.25 * N  # 102^3: just above 2^20 particles
    n = S ** 3
    x = _positions(order, S, L)
    m = torch.as_tensor(np.random.default_rng(1).uniform(0.5, 2.0, n), device="cuda") if explicit else None
    kw = {} if method == "pure_pm" else {"method": method, "split_scale": 1.5 * L / N}
    s = H.PMSolver(L, N, precision=prec, max_particles=n, **kw)
    got, ref = ([torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(3)] for _ in range(2))
    s.compute_forces(*x, m, None if explicit else 1.5, *got)
    src = s.density(*x, m, 0.0 if explicit else 1.5)
    if method == "pure_pm":
        s.gather(s.potential(src), *x, *ref)
    else:
        for f, r in zip(s.force_meshes(src), ref):
            s.interpolate(f, *x, r)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("order", ["lattice", "shuffled"])
def test_refused_position_leaves_accelerations(gpu, order):
    import torch

    import hyowon_amd as H
    S, N, L = 102, 192, 192.0
    x = _positions(order, S, L)
    x[1][12345] = float("inf")
    s = H.PMSolver(L, N, precision="fp32", max_particles=S ** 3)
    acc = [torch.ones(S ** 3, dtype=torch.float64, device="cuda") for _ in range(3)]
    with pytest.raises(ValueError, match="positions must be finite"):
        s.compute_forces(*x, None, 1.0, *acc)
    assert all(torch.equal(t, torch.ones_like(t)) for t in acc)


def test_force_in_lattice_order_costs_no_more_than_a_step(gpu):
    import torch

    import hyowon_amd as H
    S, N, L = 256, 512, 512.0
    x = _positions("lattice", S, L)
    s = H.PMSolver(L, N, precision="fp32", max_particles=S ** 3)
    acc = [torch.zeros(S ** 3, dtype=torch.float64, device="cuda") for _ in range(3)]
    a = H.ParticleState(*x, *(torch.zeros(S ** 3, dtype=torch.float32, device="cuda") for _ in range(3)))
    b = a.empty_like()

    def timed(f):
        times = []
        for _ in range(11):
            torch.cuda.synchronize()
            t = time.perf_counter()
            f()
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t)
        return sorted(times)[5]

    force, step = timed(lambda: s.compute_forces(*x, None, 1.0, *acc)), timed(lambda: s.kdk(a, b, 1.0, None, 1e-3, 1e-3))
    assert force < 1.1 * step, (force, step)
