"""Evaluations of the orders above 10 at the ends of their range: the largest
requests for shared memory under graph capture."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [31, 40])
def test_captured_steps_equal_eager(p):
    """M2M and M2L ask for up to 147 and 139 KB of shared memory per launch, in
    captured launches too."""
    import fmms_amd as fa

    pos, mass = O.plummer(600, seed=p)
    vel = np.zeros_like(pos)
    out = []
    for graph in (False, True):
        f = fa.Fmm(None, None, p=p, eps=math.inf, n_leaf=16, theta_max=0.6)
        it = fa.Integrator(f, pos, vel, mass)
        for _ in range(3):
            it.step(1e-3, steps=2, refresh_every=8, graph=graph)
        out.append(it.state())
        assert f.leapfrog_stats()["frozen_steps"] > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)
