"""fmin of every cell from block minima: the smallest f of its bodies, exactly,
at sizes around one and two blocks of 64 and of 4096 slots, and where cells'
ranges begin and end within blocks."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 4095, 4096, 4097, 9000, 20000])
def test_fmin_is_the_minimum_of_the_cells_bodies(n):
    import fmms_amd as fa

    print(f"[fmin] n={n}", flush=True)
    pos, mass = O.plummer(n, seed=n)
    g = fa.Fmm(pos, mass, p=3, eps=1e-3, n_leaf=5)
    g.run(pos, mass)
    f, fmin = g.f()
    t = g.tree()
    first, count = np.asarray(t.first, np.int64), np.asarray(t.count, np.int64)
    want = np.array([f[a:a + c].min() for a, c in zip(first, count)])
    assert np.array_equal(fmin.view(np.uint64), want.view(np.uint64))
