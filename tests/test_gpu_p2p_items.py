"""The P2P work plan against its rule, recomputed from the lists: how many items
the leaves are cut into, with the FP64 form's cap on an item's sources (default
item bound) and without it (a larger bound is the caller's choice, the mixed form
has none); and systems in which a few items are long, which are launched first."""
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

CAP = 4096


def leaf_sources(g):
    """(targets, sources, list entries) per leaf, from the P2P pairs."""
    t = g.tree()
    nt = np.asarray(t.count, np.int64)
    leaf = np.asarray(t.leaf, bool)
    s, units = nt.copy(), np.ones_like(nt)  # the leaf's own bodies
    p2p = np.asarray(g.lists()[1], np.int64)
    a, b = p2p[:, 0], p2p[:, 1]
    units += np.bincount(a, minlength=len(nt))
    off = a != b
    units += np.bincount(b[off], minlength=len(nt))
    s += np.bincount(a[off], nt[b[off]], len(nt)).astype(np.int64)
    s += np.bincount(b[off], nt[a[off]], len(nt)).astype(np.int64)
    return nt[leaf], s[leaf], units[leaf]


def leaf_items(nt, s, units, work, cap):
    m = np.maximum(1, -(-(nt * s) // work))
    if cap:
        m = np.where(s > cap, np.maximum(m, (s - 1) // cap + 1), m)
    return np.minimum(m, units)


@pytest.mark.parametrize("precision,work", [("fp64", 1 << 18), ("fp64", 1 << 15), ("fp64", 1 << 19),
                                            ("fp64", 1 << 40), ("fp32bulk", 1 << 18)])
def test_item_counts(precision, work):
    import fmms_amd as fa

    pos, mass = fa.plummer(12000, seed=5)
    kw = dict(p=3, eps=math.inf, n_leaf=48, theta_max=0.2, softening=1e-2)
    g = fa.Fmm(None, None, p2p_item_work=work, precision=precision, **kw)
    r = g.accel(pos, mass)
    capped = precision == "fp64" and work <= 1 << 18
    nt, s, units = leaf_sources(g)
    m = leaf_items(nt, s, units, work, CAP if capped else 0)
    assert (s > CAP).sum() > 50
    wc = g.work_counts()
    assert wc["p2p_items"] == m.sum() and wc["p2p_split_leaves"] == (m > 1).sum()
    if work == 1 << 40:
        assert wc["p2p_items"] == wc["nleaves"]
    if precision == "fp64":  # the same sums, cut elsewhere
        a = fa.Fmm(None, None, **kw).accel(pos, mass)
        an = np.linalg.norm(a.accel, axis=1)
        assert np.all(np.linalg.norm(r.accel - a.accel, axis=1) <= 1e-13 * an + 1e-15 * an.max())
        assert np.allclose(r.pot, a.pot, rtol=1e-13, atol=0)


# sources above which an item is long, and neighbours up to which none is
LONG = {"fp64": 2048, "fp32bulk": 8192}
SHORT_LIST = 32


@pytest.mark.parametrize("n,n_leaf,theta", [(20000, 16, 0.5), (20000, 8, 0.8), (30000, 16, 0.7)])
def test_long_items_first(n, n_leaf, theta):
    import fmms_amd as fa

    pos, mass = O.plummer(n, seed=5)
    mass = mass * np.linspace(0.5, 1.5, n)
    kw = dict(p=2, eps=math.inf, n_leaf=n_leaf, theta_max=theta, softening=1e-2)
    out = {}
    for precision in ("fp64", "fp32bulk"):
        g = fa.Fmm(None, None, precision=precision, **kw)
        out[precision] = g.accel(pos, mass)
        nt, s, units = leaf_sources(g)
        m = leaf_items(nt, s, units, 1 << 18, CAP if precision == "fp64" else 0)
        nlong = m[(units - 1 > SHORT_LIST) & (s // m > LONG[precision])].sum()
        assert g.work_counts()["p2p_items"] == m.sum()
        assert 0 < nlong and 16 * nlong <= m.sum()  # few: launched first
    orc = O.OracleFmm(pos, mass, **kw)
    a_ref, pot_ref = orc.run(pos, mass)
    an = np.linalg.norm(a_ref, axis=1)
    # the same sums in another order: the suite's FP64 bars, and the mixed form's
    r, m = out["fp64"], out["fp32bulk"]
    assert np.all(np.linalg.norm(r.accel - a_ref, axis=1) <= 1e-11 * an + 1e-13 * an.max())
    assert np.allclose(r.pot, pot_ref, rtol=1e-11, atol=0)
    assert np.all(np.linalg.norm(m.accel - r.accel, axis=1) <= 2e-5 * an + 2e-6 * an.max())
