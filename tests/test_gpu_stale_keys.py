"""Synchronous steps whose carried keys are stale (the positions changed between
the calls): routed afresh, in one box and in several, on meshes where the host
looks at the keys' verdict during the deposit (256^3) and below; and no transform
is spent on the stale routing of a large mesh."""
import time

import numpy as np
import pytest

from conftest import clumpy_particles

pytestmark = pytest.mark.gpu


def _state(H, pos, mom, prec):
    a = H.ParticleState.from_numpy(pos, mom, precision=prec)
    return a, a.empty_like()


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N,boxes", [(16, 1), (32, 3), (256, 1), (128, 8)])
def test_stale_step_equals_fresh_one(gpu, prec, N, boxes):
    import hyowon_amd as H
    import torch
    L, n = 1.5 * N, 2000
    pos = np.concatenate([clumpy_particles(n, L, 9 + b) for b in range(boxes)], axis=1)
    mom = np.random.default_rng(boxes).normal(0, 5.0, pos.shape)

    def run(reuse):
        s = H.PMSolver(L, N, precision=prec, max_particles=n * boxes, boxes=boxes)
        a, b = _state(H, pos, mom, prec)
        s.kdk(a, b, 1.0, None, 0.01, 0.02, reuse_keys=reuse)
        b.y.add_(0.37 * L).remainder_(L)
        b.x[::7] += 2.0 * L / N
        s.kdk(b, a, 1.0, 0.01, 0.01, 0.02, reuse_keys=reuse)  # stale where reuse
        s.kdk(a, b, 1.0, 0.01, 0.01, 0.02, reuse_keys=reuse)  # and carried again
        return [b.x, b.y, b.z, b.px, b.py, b.pz]

    for u, v in zip(run(True), run(False)):
        assert torch.equal(u, v)


@pytest.mark.parametrize("N", [32, 256])
def test_stale_and_not_finite_is_refused(gpu, N):
    import hyowon_amd as H
    import torch
    L, n = 1.0 * N, 2000
    a, b = _state(H, clumpy_particles(n, L, 4), np.zeros((3, n)), "fp32")
    s = H.PMSolver(L, N, precision="fp32", max_particles=n)
    s.kdk(a, b, 1.0, None, 0.01, 0.02)
    b.x.add_(0.5 * L)
    b.z[17] = float("nan")
    before = [t.clone() for t in (a.x, a.px)]
    with pytest.raises(ValueError, match="positions must be finite"):
        s.kdk(b, a, 1.0, 0.01, 0.01, 0.02, reuse_keys=True)
    assert all(torch.equal(u, v) for u, v in zip((a.x, a.px), before))


def test_stale_keys_cost_no_transform(gpu):
    """512^3 binary32 mesh, 2^21 particles: the transform is most of the call, so a
    second one shows as a factor near 2 over a call that routes from scratch."""
    import hyowon_amd as H
    import torch
    N, L, n = 512, 512.0, 1 << 21
    rng = np.random.default_rng(1)
    a, b = _state(H, rng.uniform(0.0, L, (3, n)), np.zeros((3, n)), "fp32")
    s = H.PMSolver(L, N, precision="fp32", max_particles=n)

    def timed(reuse):
        s.kdk(a, b, 1.0, None, 1e-3, 1e-3)
        b.x.add_(3.0).remainder_(L)
        torch.cuda.synchronize()
        t = time.perf_counter()
        s.kdk(b, a, 1.0, None, 1e-3, 1e-3, reuse_keys=reuse)
        torch.cuda.synchronize()
        return time.perf_counter() - t

    timed(True)
    fresh, stale = (sorted(timed(r) for _ in range(9))[4] for r in (False, True))
    assert stale < 1.6 * fresh, (stale, fresh)
