"""The error-controlled walk at every order it is compiled for and one beyond:
the pair sets are the oracle's, and the decisions differ from the theta-only
walk's (so the estimate decided some)."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", range(1, 13))
def test_error_mac_lists_match_oracle(p):
    import fmms_amd as fa

    print(f"[mac] p={p}", flush=True)
    n = 1500
    pos, mass = O.plummer(n, seed=40 + p)
    mass = mass * np.linspace(0.5, 1.5, n)
    kw = dict(p=p, eps=10.0 ** (-1 - p / 2), n_leaf=8, theta_max=1.0)
    orc = O.OracleFmm(pos, mass, **kw)
    orc.run(pos, mass)
    g = fa.Fmm(None, None, **kw)
    g.accel(pos, mass)
    m2l, p2p = g.lists()
    assert sorted(map(tuple, m2l)) == sorted(map(tuple, orc.m2l_pairs()))
    assert sorted(map(tuple, p2p)) == sorted(map(tuple, orc.p2p_pairs()))
    th = fa.Fmm(None, None, **{**kw, "eps": math.inf})
    th.accel(pos, mass)
    assert 0 < len(m2l) and len(p2p) > len(th.lists()[1])
