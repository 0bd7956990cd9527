"""The walk's rounds (walk.hip): frontiers smaller than a batch and larger
than one per block, lists that outgrow the first buffers (a round halts and
resumes), and an empty walk; the pair sets are the oracle's."""
import math

import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_leaf,theta", [(1, 4, 0.5), (3, 1, 0.9), (300, 8, 0.5), (6000, 8, 0.15),
                                            (30000, 64, 0.3)])
def test_lists_match_oracle(n, n_leaf, theta):
    import fmms_amd as fa

    pos, mass = O.plummer(n, seed=n % 89)
    kw = dict(p=2, eps=math.inf, n_leaf=n_leaf, theta_max=theta)
    orc = O.OracleFmm(pos, mass, **kw)
    orc.run(pos, mass)
    g = fa.Fmm(None, None, **kw)
    for _ in range(2):  # the second walk starts with the grown buffers
        g.accel(pos, mass)
        m2l, p2p = g.lists()
        assert sorted(map(tuple, m2l)) == sorted(map(tuple, orc.m2l_pairs()))
        assert sorted(map(tuple, p2p)) == sorted(map(tuple, orc.p2p_pairs()))
