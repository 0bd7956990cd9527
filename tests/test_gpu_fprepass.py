"""f pre-pass (upward.hip) bit for bit against the oracle on both sides of
the line between four lanes and one lane per body, at counts that fill no
wave, and with coincident bodies and massless ones."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 17, 1003, 131072, 131073])
def test_f_bit_exact(n):
    import fmms_amd as fa

    pos, mass = O.plummer(n, seed=n % 97)
    if n > 10:
        pos[3] = pos[7]
        mass[5] = 0.0
    kw = dict(p=2, eps=1e-2, n_leaf=13)
    orc = O.OracleFmm(pos, mass, **kw)
    orc.run(pos, mass)
    g = fa.Fmm(pos, mass, **kw)
    g.run(pos, mass)
    f, fmin = g.f()
    assert np.array_equal(f.view(np.uint64), orc.f().view(np.uint64))
    assert np.array_equal(fmin.view(np.uint64), orc.fmin().view(np.uint64))
