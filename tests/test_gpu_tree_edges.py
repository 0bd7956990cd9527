"""Trees built from the sorted keys (tree.hip) and the sorts behind them, bit
for bit against the oracle where they change route: one sort tile, tiles that
sum the histogram themselves and scanned ones (2048 and 131072 elements),
leaf capacities of one, odd and even, a capacity that just holds and just
overflows the input, and runs of coincident bodies longer than a leaf."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [(1, 1), (2, 1), (16, 16), (17, 16), (2048, 7), (2049, 8), (5000, 1), (131072, 33),
         (131073, 32)]


@pytest.mark.parametrize("n,n_leaf", CASES)
@pytest.mark.parametrize("dup", [False, True])
def test_tree_bit_exact(n, n_leaf, dup):
    import fmms_amd as fa

    pos, mass = O.plummer(n, seed=7 + n % 11)
    if dup and n > 2:  # a run of coincident bodies and a run on one line
        k = max(1, min(n // 3, 3 * n_leaf))
        pos[:k] = pos[0]
        pos[k:2 * k, 1:] = pos[k, 1:]
    orc = O.OracleFmm(pos, mass, p=2, eps=1e-2, n_leaf=n_leaf)
    g = fa.Fmm(pos, mass, p=2, eps=1e-2, n_leaf=n_leaf)
    tg, to = g.tree(), orc.tree()
    for name in ("order", "keys", "first", "count", "children", "leaf", "level"):
        assert np.array_equal(getattr(tg, name), getattr(to, name)), name
    for name in ("cen", "mass", "rho"):
        a, b = getattr(tg, name), getattr(to, name)
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), name
