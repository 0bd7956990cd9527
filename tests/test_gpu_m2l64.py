"""FP64 M2L of the templated orders (m2l_kernel.h) against the oracle, at
every order (row staging up to p = 8, rows read directly above, accumulators
split over two waves from p = 9) and at the chunk lengths where a wave's
lanes run different trip counts: single sources, a length that divides no
list, and chunks longer than any list (fewer chunks than lanes)."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", range(1, 11))
@pytest.mark.parametrize("chunk,soft,n", [(1, 0.0, 300), (7, 1e-3, 1100), (1024, 0.0, 700)])
def test_fp64_m2l_matches_oracle(p, chunk, soft, n):
    import fmms_amd as fa

    pos, mass = O.plummer(n, seed=300 + p)
    mass = mass * np.linspace(0.5, 1.5, n)  # dipoles and odd orders of every size
    kw = dict(p=p, eps=math.inf, n_leaf=12, theta_max=0.7, softening=soft)
    orc = O.OracleFmm(pos, mass, **kw)
    a_ref, pot_ref = orc.run(pos, mass)
    g = fa.Fmm(pos, mass, m2l_chunk=chunk, **kw)
    r = g.run(pos, mass)
    assert len(g.lists()[0]) > 0
    # the same sums in another order: the suite's FP64 bars
    an = np.linalg.norm(a_ref, axis=1)
    assert np.all(np.linalg.norm(r.accel - a_ref, axis=1) <= 1e-11 * an + 1e-13 * an.max())
    assert np.allclose(r.pot, pot_ref, rtol=1e-11, atol=0)
    lg, lo = g.locals(), orc.locals()
    assert np.abs(lg - lo).max() <= 1e-10 * np.abs(lo).max()
