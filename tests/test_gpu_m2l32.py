"""FP32 M2L of the mixed form against the FP64 M2L at every templated order
(rows staged through LDS for p = 3..8, read directly for the others) and at the
chunk lengths where a wave's lanes run different trip counts: single sources, a
length that divides no list, and chunks longer than any list (fewer chunks than
lanes)."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", range(1, 11))
@pytest.mark.parametrize("chunk,soft,n", [(1, 1e-3, 2000), (7, 1e-3, 3000), (1024, 1e-3, 600)])
def test_fp32_m2l_matches_fp64(p, chunk, soft, n):
    import fmms_amd as fa

    print(f"[m2l32] p={p} chunk={chunk} n={n}", flush=True)
    pos, mass = O.plummer(n, seed=500 + p)
    kw = dict(p=p, eps=math.inf, n_leaf=16, theta_max=0.5, softening=soft)
    g64 = fa.Fmm(pos, mass, **kw)
    g64.run(pos, mass)
    g32 = fa.Fmm(pos, mass, precision="fp32bulk", m2l_chunk=chunk, **kw)
    g32.run(pos, mass)
    m2l = np.asarray(g32.lists()[0])
    assert len(m2l) > 0
    longest = np.bincount(m2l.ravel()).max()  # sources of one target, both directions
    l64, l32 = g64.locals(), g32.locals()
    t = g64.tree()
    n_of = np.concatenate([[k] * (2 * k + 1) for k in range(p + 1)])
    w = np.maximum(t.rho, 1e-12)[:, None] ** n_of[None, :]
    num, den = (np.abs(l32 - l64) * w).sum(1), (np.abs(l64) * w).sum(1)
    rel = num[den > 0] / den[den > 0]
    # the suite's bar for FP32 sums of up to 32 sources, growing with their number
    assert rel.max() < 2e-5 * max(1.0, min(chunk, longest) / 32), rel.max()
