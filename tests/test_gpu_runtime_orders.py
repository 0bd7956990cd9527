"""Evaluations of the orders above 10: the rounding of the rotation M2L where the
direct convolution is the reference (orders below 20), the last orders (six
K-steps, three 16-row tiles, the largest requests for shared memory), and those
under graph capture."""
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


def _run(p, n, theta, soft, clump=False):
    import fmms_amd as fa

    pos, mass = O.plummer(n, seed=70 + p)
    mass = mass * np.linspace(0.5, 1.5, n)
    if clump:
        pos[: n // 2] = pos[: n // 2] * 1e-3 + [3.0, 1.0, -2.0]
    kw = dict(p=p, eps=math.inf, n_leaf=16, theta_max=theta, softening=soft)
    a_ref, pot_ref = O.OracleFmm(pos, mass, **kw).run(pos, mass)
    g = fa.Fmm(pos, mass, **kw)
    r = g.run(pos, mass)
    assert len(g.lists()[0]) > 0
    return r, a_ref, pot_ref, np.linalg.norm(a_ref, axis=1)


@pytest.mark.parametrize("p", range(11, 20))
@pytest.mark.parametrize("clump", [False, True])
def test_rotation_rounds_like_the_convolution(p, clump):
    """The oracle convolves below p = 20. Both routes' far forces are within 5e-15
    of the 80-bit sum of the same expansions (median 1e-16 by rotation, 3e-16 by
    convolution), so an error that had grown with the rotation would show far
    below the 1e-9 the two methods are held to."""
    r, a_ref, pot_ref, an = _run(p, 700, 0.7, 0.0, clump)
    assert np.all(np.linalg.norm(r.accel - a_ref, axis=1) <= 1e-13 * an + 1e-15 * an.max())
    assert np.allclose(r.pot, pot_ref, rtol=1e-13, atol=0)


@pytest.mark.parametrize("p", [39, 40])
@pytest.mark.parametrize("soft", [0.0, 2e-3])
def test_last_orders_match_oracle(p, soft):
    # two rotations in other operation orders: the methods' own contract
    r, a_ref, pot_ref, an = _run(p, 500, 0.7, soft)
    assert np.all(np.linalg.norm(r.accel - a_ref, axis=1) <= 1e-9 * an + 1e-11 * an.max())
    assert np.allclose(r.pot, pot_ref, rtol=1e-9, atol=0)
