"""Forces gathered in record order: the same bits as the particle-order
gather and interpolation of the same meshes, for shuffled and sorted particles,
tile edges of 16, 12 and 8, counts around a workgroup, explicit masses and
several boxes."""
import numpy as np
import pytest

from conftest import clumpy_particles

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda:0")


def _zeros(n):
    import torch
    return [torch.zeros(n, dtype=torch.float64, device="cuda:0") for _ in range(3)]


@pytest.mark.parametrize("N,L,n", [(8, 8.0, 1), (12, 30.0, 255), (24, 24.0, 257), (32, 32.0, 20000), (64, 96.0, 100000)])
@pytest.mark.parametrize("order", ["sorted", "shuffled"])
@pytest.mark.parametrize("explicit", [False, True])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_force_equals_particle_order_gather(gpu, N, L, n, order, explicit, prec):
    import hyowon_amd as H
    pos = clumpy_particles(n, L, N)
    idx = np.lexsort(pos[::-1]) if order == "sorted" else np.random.default_rng(n).permutation(n)
    x = [_dev(p[idx]) for p in pos]
    m = _dev(np.random.default_rng(1).uniform(0.5, 2.0, n)) if explicit else None
    s = H.PMSolver(L, N, precision=prec, max_particles=n)
    got, ref = _zeros(n), _zeros(n)
    s.compute_forces(*x, m, None if explicit else 1.5, *got)
    s.gather(s.potential(s.density(*x, m, 0.0 if explicit else 1.5)), *x, *ref)
    for a, b in zip(got, ref):
        assert np.array_equal(a.cpu().numpy(), b.cpu().numpy())


@pytest.mark.parametrize("N,L,n", [(12, 30.0, 257), (48, 48.0, 30000)])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_treepm_force_equals_interpolation(gpu, N, L, n, prec):
    import hyowon_amd as H
    x = [_dev(p) for p in clumpy_particles(n, L, N)]
    s = H.PMSolver(L, N, precision=prec, max_particles=n, method="treepm_long_range", split_scale=1.5 * L / N)
    got, ref = _zeros(n), _zeros(n)
    s.compute_forces(*x, None, 1.5, *got)
    for f, r in zip(s.force_meshes(s.density(*x, None, 1.5)), ref):
        s.interpolate(f, *x, r)
    for a, b in zip(got, ref):
        assert np.array_equal(a.cpu().numpy(), b.cpu().numpy())


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_batched_boxes_equal_single_ones(gpu, prec):
    import hyowon_amd as H
    import torch
    N, L, n, boxes = 16, 16.0, 300, 3
    pos = np.stack([clumpy_particles(n, L, 7 + b) for b in range(boxes)])
    s = H.PMSolver(L, N, precision=prec, max_particles=n * boxes, boxes=boxes)
    got = _zeros(n * boxes)
    s.compute_forces(*(_dev(pos[:, d].reshape(-1)) for d in range(3)), None, 1.0, *got)
    one = H.PMSolver(L, N, precision=prec, max_particles=n)
    for b in range(boxes):
        ref = _zeros(n)
        one.compute_forces(*(_dev(p) for p in pos[b]), None, 1.0, *ref)
        for a, r in zip(got, ref):
            assert torch.equal(a[b * n:(b + 1) * n], r)
