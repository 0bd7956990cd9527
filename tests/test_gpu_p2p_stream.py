"""P2P source streams and work items (near.hip) at their edges: leaves of one
body (64 ranges in a tile), streams of more than 256 ranges, leaves cut at the
FP64 form's sources-per-item cap, long items launched first, and totals that
fill a last tile exactly or by one body. Nearly everything is near field
(theta 0.05); the oracle evaluates the same lists."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_leaf", [(1, 1), (2, 1), (64, 1), (65, 1), (320, 1), (700, 3),
                                      (4096, 16), (4097, 40), (9000, 24)])
def test_near_field_matches_oracle(n, n_leaf):
    import fmms_amd as fa

    pos, mass = fa.plummer(n, seed=n)
    mass = mass * np.linspace(0.5, 1.5, n)
    if n > 100:
        pos[0] = [30.0, -20.0, 25.0]  # a sparse leaf that sees every other body
    kw = dict(p=2, eps=math.inf, n_leaf=n_leaf, theta_max=0.05, softening=1e-2)
    orc = O.OracleFmm(pos, mass, **kw)
    a_ref, pot_ref = orc.run(pos, mass)
    g = fa.Fmm(None, None, **kw)
    r = g.accel(pos, mass)
    if n >= 9000:
        wc = g.work_counts()
        assert wc["p2p_items"] > wc["nleaves"], wc
    an = np.linalg.norm(a_ref, axis=1)
    # the same sums in another order: the suite's FP64 bars
    assert np.all(np.linalg.norm(r.accel - a_ref, axis=1) <= 1e-11 * an + 1e-13 * an.max())
    assert np.allclose(r.pot, pot_ref, rtol=1e-11, atol=0)
    if n > 1:
        m = fa.Fmm(None, None, precision="fp32bulk", **kw).accel(pos, mass)
        assert np.all(np.linalg.norm(m.accel - r.accel, axis=1) <= 2e-5 * an + 2e-6 * an.max())
