"""Rotation M2L of the runtime orders (p > 10, m2l_rot.hip) against the
oracle (naive convolution below p = 20, rotation from there) at the edges of
its tiles: one and two K-steps and 16-row tiles, 16 and 8 pairs per batch,
chunks with a partly filled last batch, the softened kernel, targets on the
z axis of their sources, and a frozen step replayed from a graph."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fa():
    import fmms_amd

    return fmms_amd


def _check(fa, pos, mass, p, theta, soft, n_leaf):
    orc = O.OracleFmm(pos, mass, p=p, eps=math.inf, n_leaf=n_leaf, theta_max=theta, softening=soft)
    a_ref, pot_ref = orc.run(pos, mass)
    g = fa.Fmm(pos, mass, p=p, eps=math.inf, n_leaf=n_leaf, theta_max=theta, softening=soft)
    r = g.run(pos, mass)
    assert len(g.lists()[0]) > 0
    # two summation orders of the same expansions: the reference's own
    # rotation-vs-naive contract (1e-9), 1e-11 at the orders near the templated ones
    rel = 1e-11 if p <= 12 else 1e-9
    an = np.linalg.norm(a_ref, axis=1)
    assert np.all(np.linalg.norm(r.accel - a_ref, axis=1) <= rel * an + 1e-2 * rel * an.max())
    assert np.allclose(r.pot, pot_ref, rtol=rel, atol=0)


@pytest.mark.parametrize("p", [11, 14, 15, 16, 22, 23, 31, 32, 33])
@pytest.mark.parametrize("soft", [0.0, 2e-3])
def test_orders_match_oracle(fa, p, soft):
    pos, mass = O.plummer(500, seed=60 + p)
    _check(fa, pos, mass, p, 0.7, soft, 16)


def test_pairs_along_the_z_axis(fa):
    """Leaves of single bodies stacked on one axis: alpha is undefined there
    (0 by convention) and beta is 0 or pi."""
    pos = np.zeros((24, 3))
    pos[:, 2] = np.linspace(0.0, 1.0, 24) ** 1.5
    mass = np.full(24, 1.0 / 24)
    _check(fa, pos, mass, 13, 0.9, 0.0, 1)


def test_frozen_graph_replays_equal_eager(fa):
    pos, mass = O.plummer(800, seed=91)
    vel = np.zeros_like(pos)
    out = []
    for graph in (False, True):
        f = fa.Fmm(None, None, p=12, eps=math.inf, n_leaf=16, theta_max=0.6)
        it = fa.Integrator(f, pos, vel, mass)
        for _ in range(3):
            it.step(1e-3, steps=2, refresh_every=8, graph=graph)
        out.append(it.state())
        assert f.leapfrog_stats()["frozen_steps"] > 0
    for a, b in zip(*out):
        assert np.array_equal(a, b)
