"""Gather schedules of lattices whose side is no multiple of 256: every number of
rows per column tile (narrow columns at the upper edges, short last chunks)
gives the bits of the particle-order schedule, in steps that carry keys and in
asynchronous ones that carry records."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("S,N", [(56, 48), (61, 64), (64, 32), (120, 96)])
def test_wave_schedule_keeps_bits(gpu, prec, S, N):
    import hyowon_amd as H
    L, n = 1.5 * N, S ** 3
    rng = np.random.default_rng(S)
    q = (np.arange(S) + 0.5) * (L / S)
    pos = np.mod(np.stack([a.ravel() for a in np.meshgrid(q, q, q, indexing="ij")]) + rng.normal(0, 0.5, (3, n)), L)
    mom = rng.normal(0, 5.0, (3, n))

    def run(rows, sync):
        s = H.PMSolver(L, N, precision=prec, max_particles=n)
        s.set_gather_rows(rows)
        a = H.ParticleState.from_numpy(pos, mom, precision=prec)
        b = a.empty_like()
        for i in range(3):
            s.kdk(a, b, 1.0, 0.01 if i else None, 0.01, 0.02, reuse_keys=True, asynchronous=not sync)
            a, b = b, a
        s.check()
        out = [t.cpu().numpy() for t in (a.x, a.y, a.z, a.px, a.py, a.pz)]
        s.close()
        return out

    ref = run(0, True)
    for rows, sync in [(None, True), (1, True), (8, False), (None, False), (4096, False)]:
        for u, v in zip(run(rows, sync), ref):
            assert np.array_equal(u, v), (rows, sync)
