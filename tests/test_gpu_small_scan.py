"""Bucket scans on both sides of the one-workgroup limit (16384 buckets: four boxes
of a 128^3 mesh), and synchronous calls that read their status once, at the
end: a failed deposit leaves outputs and accelerations as they were."""
import numpy as np
import pytest

from conftest import clumpy_particles

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda:0")


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N,boxes", [(16, 1), (128, 4), (128, 5)])
def test_batched_boxes_equal_single_ones(gpu, prec, N, boxes):
    import hyowon_amd as H
    import torch
    L, n = 1.5 * N, 4096
    pos = np.stack([clumpy_particles(n, L, 3 + b) for b in range(boxes)])
    mom = np.random.default_rng(boxes).normal(0, 5.0, pos.shape)

    def run(p, m, nb):
        s = H.PMSolver(L, N, precision=prec, max_particles=p.shape[1], boxes=nb)
        a = H.ParticleState.from_numpy(p, m, precision=prec)
        b = a.empty_like()
        for i in range(3):
            s.kdk(a, b, 1.0, 0.01 if i else None, 0.01, 0.02, reuse_keys=True, asynchronous=i == 1)
            a, b = b, a
        s.check()
        return [a.x, a.y, a.z, a.px, a.py, a.pz]

    got = run(pos.transpose(1, 0, 2).reshape(3, -1), mom.transpose(1, 0, 2).reshape(3, -1), boxes)
    for b in range(boxes):
        for u, v in zip(got, run(pos[b], mom[b], 1)):
            assert torch.equal(u[b * n:(b + 1) * n], v)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_failed_deposit_leaves_state(gpu, prec):
    import hyowon_amd as H
    import torch
    N, L, n = 32, 32.0, 5000
    pos = clumpy_particles(n, L, 1)
    bad = pos.copy()
    bad[1, 137] = np.nan
    mom = np.zeros((3, n))
    s = H.PMSolver(L, N, precision=prec, max_particles=n)
    a, b = (H.ParticleState.from_numpy(p, mom, precision=prec) for p in (bad, pos))
    before = [t.clone() for t in (b.x, b.y, b.z, b.px, b.py, b.pz)]
    with pytest.raises(ValueError, match="positions must be finite"):
        s.kdk(a, b, 1.0, None, 0.01, 0.02)
    for u, v in zip((b.x, b.y, b.z, b.px, b.py, b.pz), before):
        assert torch.equal(u, v)
    acc = [torch.ones(n, dtype=torch.float64, device="cuda:0") for _ in range(3)]
    with pytest.raises(ValueError, match="positions must be finite"):
        s.compute_forces(a.x, a.y, a.z, None, 1.0, *acc)
    assert all(torch.equal(t, torch.ones_like(t)) for t in acc)
    # the context recovers
    s.compute_forces(b.x, b.y, b.z, None, 1.0, *acc)
    assert all(torch.isfinite(t).all() and not torch.equal(t, torch.ones_like(t)) for t in acc)
