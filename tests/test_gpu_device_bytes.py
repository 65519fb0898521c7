"""Device memory of a context per particle of capacity (hy_pm_info.device_bytes): the
keys, ranks, records, forces, deposit scratch and binary64 job list that calls use."""
import pytest

pytestmark = pytest.mark.gpu

# binary32: key and rank 8, records 34 (two and an eighth of 16), mass 4, force 12,
# scratch 16; binary64: key and rank 8, record 32, mass 8, force 24, scratch 16, jobs 0.75
PER_PARTICLE = {"fp32": 74.0, "fp64": 88.75}


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_bytes_per_particle(gpu, prec):
    import hyowon_amd as H
    # enough tiles that the job list is bounded by the particles, not by them
    small, large = (H.PMSolver(128.0, 128, precision=prec, max_particles=n) for n in (160000, 320000))
    got = (large.info().device_bytes - small.info().device_bytes) / 160000
    assert got == pytest.approx(PER_PARTICLE[prec], abs=0.01)
