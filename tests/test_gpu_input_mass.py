"""The exact sum of explicit particle masses formed on the device
(hy_pm_get_info's last_input_mass) against the oracle's correctly rounded sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _masses(kind, n):
    rng = np.random.default_rng(n)
    if kind == "narrow":
        return rng.uniform(0.5, 2.0, n)
    if kind == "wide":  # more binary orders than a thread's digit window holds
        return np.ldexp(rng.uniform(0.5, 1.0, n), rng.integers(-200, 200, n))
    m = rng.uniform(0.5, 2.0, n)  # zeros, ties: sums whose last bits decide
    m[::2] = 0.0
    m[1::4] = 1.0 + 2.0 ** -52
    m[0] = 2.0 ** 40
    return m


@pytest.mark.parametrize("n", [1, 2, 63, 257, 1025, 300001])
@pytest.mark.parametrize("kind", ["narrow", "wide", "ties"])
def test_input_mass_is_the_exact_sum(gpu, oracle_mod, kind, n):
    import torch

    import hyowon_amd as H
    N, L = 16, 16.0
    m = _masses(kind, n)
    pos = np.random.default_rng(n + 1).uniform(0.0, L, (3, n))
    s = H.PMSolver(L, N, precision="fp64", max_particles=n)
    t = [torch.as_tensor(p, device=gpu) for p in pos]
    for _ in range(2):  # the counters are left clean by a call
        s.density(*t, torch.as_tensor(m, device=gpu), 0.0)
        want = float(oracle_mod.lib().or_exact_sum(m.ctypes.data_as(oracle_mod._pd), n))
        assert s.info().last_input_mass == want


@pytest.mark.parametrize("bad", [np.nan, np.inf, -1.0])
def test_invalid_mass_is_refused_and_the_next_call_is_clean(gpu, bad):
    import torch

    import hyowon_amd as H
    n, N, L = 1000, 16, 16.0
    rng = np.random.default_rng(3)
    t = [torch.as_tensor(p, device=gpu) for p in rng.uniform(0.0, L, (3, n))]
    m = rng.uniform(0.5, 2.0, n)
    wrong = m.copy()
    wrong[777] = bad
    s = H.PMSolver(L, N, precision="fp64", max_particles=n)
    with pytest.raises(ValueError):
        s.density(*t, torch.as_tensor(wrong, device=gpu), 0.0)
    s.density(*t, torch.as_tensor(m, device=gpu), 0.0)
    assert abs(s.info().last_input_mass - m.sum()) <= 1e-12 * m.sum()
