"""The launch variants that a new context starts with, on every size that has several,
are within a quarter of the fastest that the autotuner times (its times for one
variant repeat to a few percent; the smallest passes, 10 us, to a tenth)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("N", [192, 256, 384, 512, 1024])
def test_start_plan_is_near_the_fastest(gpu, N, prec):
    import hyowon_amd as H
    s = H.PMSolver(float(N), N, precision=prec, max_particles=1)
    start = s.tuning()["variant"]
    ms = s.autotune(reps=5)["pass_ms"]
    for name, v in start.items():
        assert ms[name][v] <= 1.25 * min(ms[name]), (name, v, ms[name])
