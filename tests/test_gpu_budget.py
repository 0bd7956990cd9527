"""Contexts with a device-memory budget: every evaluation below has been
accepted within the stated bytes since before its scratch buffers (source rows
of the M2L, chunk partials of the orders above 10, partial sums of cut leaves)
were introduced, so it has to go through within them, and to give what a context
without a budget gives."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(n, budget, **kw):
    import fmms_amd as fa

    pos, mass = fa.plummer(n, seed=1)
    mass = mass * np.linspace(0.5, 1.5, n)
    free = fa.Fmm(None, None, **kw)
    tight = fa.Fmm(None, None, hbm_budget_bytes=budget, **kw)
    a = free.accel(pos, mass)
    b = tight.accel(pos, mass)
    assert tight.device_bytes() <= budget
    return a, b, tight.run_frozen(pos, mass)


# short lists at the higher templated orders: no idle list buffer holds the rows
@pytest.mark.parametrize("n,p,eps,theta,n_leaf,budget", [
    (200, 8, 1e-5, 1.0, 16, 648296),
    (1000, 10, 1e-5, 1.0, 8, 5577070),
    (5000, 10, math.inf, 0.9, 8, 18877066),
    (30000, 9, math.inf, 0.9, 1, 260903322),
    (30000, 10, math.inf, 0.9, 8, 112076136),
])
def test_source_rows(n, p, eps, theta, n_leaf, budget):
    free, tight, frozen = _pair(n, budget, p=p, eps=eps, theta_max=theta, n_leaf=n_leaf)
    assert np.array_equal(free.accel, tight.accel) and np.array_equal(free.pot, tight.pot)
    assert np.array_equal(free.accel, frozen.accel) and np.array_equal(free.pot, frozen.pot)


# orders above 10: the chunk partials do not fit at once and run in slices
@pytest.mark.parametrize("n,p,eps,theta,n_leaf,precision,budget", [
    (200, 16, math.inf, 0.7, 8, "fp64", 1507892),
    (1000, 24, math.inf, 0.5, 64, "fp64", 2635976),
    (5000, 16, math.inf, 0.5, 32, "fp64", 13126196),
    (5000, 40, math.inf, 0.5, 64, "fp64", 21893620),
    (30000, 12, 1e-6, 1.0, 16, "fp64", 102337458),
    (30000, 12, math.inf, 0.5, 64, "fp32bulk", 41461066),
    (30000, 16, math.inf, 0.5, 32, "fp64", 91418884),
    (30000, 24, math.inf, 0.5, 64, "fp64", 70305818),
])
def test_rotation_partials(n, p, eps, theta, n_leaf, precision, budget):
    free, tight, frozen = _pair(n, budget, p=p, eps=eps, theta_max=theta, n_leaf=n_leaf,
                                precision=precision,
                                softening=1e-3 if precision == "fp32bulk" else 0.0)
    assert np.array_equal(free.accel, tight.accel) and np.array_equal(free.pot, tight.pot)
    assert np.array_equal(free.accel, frozen.accel) and np.array_equal(free.pot, frozen.pot)
