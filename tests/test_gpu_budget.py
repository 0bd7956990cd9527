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


# mostly near field: leaves cut at the FP64 form's cap on an item's sources; with
# a budget that only holds the plan without the cap the sums are cut elsewhere
@pytest.mark.parametrize("n,p,theta,n_leaf,budget,same", [
    (20000, 1, 0.05, 32, 131047136, True),
    (40000, 2, 0.02, 64, 149665794, True),
    (40000, 3, 0.1, 96, 76462492, True),
    (50000, 12, 0.2, 64, 231556320, True),
    (12000, 2, 0.02, 128, 7459156, True),
    (40000, 2, 0.02, 192, 42340338, False),
])
def test_cut_leaves(n, p, theta, n_leaf, budget, same):
    free, tight, frozen = _pair(n, budget, p=p, eps=math.inf, theta_max=theta, n_leaf=n_leaf,
                                softening=1e-2 if n == 12000 else 0.0)
    assert np.array_equal(tight.accel, frozen.accel) and np.array_equal(tight.pot, frozen.pot)
    if same:
        assert np.array_equal(free.accel, tight.accel) and np.array_equal(free.pot, tight.pot)
    else:  # the same sums in another order
        an = np.linalg.norm(free.accel, axis=1)
        assert np.all(np.linalg.norm(tight.accel - free.accel, axis=1) <= 1e-13 * an + 1e-15 * an.max())
        assert np.allclose(tight.pot, free.pot, rtol=1e-13, atol=0)
