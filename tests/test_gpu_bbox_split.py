"""Boxes of an ensemble's systems: systems much larger and smaller than the mean
(several blocks each, most of them empty for the small ones), exactly one body,
and more systems than blocks (one block each). Every system's results are its
standalone evaluation's bit for bit, so its box is."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1, 40000, 2, 257, 256], [3, 5] * 550])
def test_systems_keep_their_boxes(sizes):
    import fmms_amd as fa

    print(f"[bbox] {len(sizes)} systems, {sum(sizes)} bodies", flush=True)
    rng = np.random.default_rng(len(sizes))
    pos = [rng.standard_normal((k, 3)) * rng.uniform(0.1, 10) + rng.standard_normal(3) for k in sizes]
    mass = [rng.uniform(0.5, 1.5, k) for k in sizes]
    kw = dict(p=4, eps=math.inf, n_leaf=16, theta_max=0.5, softening=1e-2)
    g = fa.Fmm(None, None, **kw)
    off = g.set_systems(sizes)
    r = g.accel(np.concatenate(pos), np.concatenate(mass))
    one = fa.Fmm(None, None, **kw)
    for i in list(range(6)) + [len(sizes) // 2, len(sizes) - 1]:
        if i >= len(sizes):
            continue
        a, b = int(off[i]), int(off[i + 1])
        ri = one.accel(pos[i], mass[i])
        assert np.array_equal(r.accel[a:b].view(np.uint64), ri.accel.view(np.uint64)), i
        assert np.array_equal(r.pot[a:b].view(np.uint64), ri.pot.view(np.uint64)), i
