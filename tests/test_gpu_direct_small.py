"""Direct sums over one range of sources, which the blocks write as they are
(fewer than 16384 bodies): few bodies with many targets, groups of four and
single targets, a last group that is not full, and outputs left out."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nt", [(1, 2050), (2, 1), (12, 4413), (257, 2049), (300, 40),
                                  (16383, 2047), (16384, 2048)])
def test_one_range_against_extended_precision(n, nt):
    import fmms_amd as fa
    from fmms_amd import hip

    print(f"[direct] n={n} nt={nt}", flush=True)
    rng = np.random.default_rng(n + nt)
    pos, mass = rng.standard_normal((n, 3)), rng.uniform(0.5, 1.5, n)
    ids = rng.integers(0, n, nt).astype(np.uint32)
    bufs = [hip.DeviceArray.from_host(x) for x in (pos, mass, ids)]
    a, p, f, a2 = (hip.DeviceArray(s) for s in ((nt, 3), (nt,), (nt,), (nt, 3)))
    call = fa.lib().fmmh_direct_sampled_noalloc
    args = (n, bufs[0].ptr, bufs[1].ptr, 1e-2, nt, bufs[2].ptr)
    assert call(*args, a.ptr, p.ptr, f.ptr, None) == fa.FMMH_OK
    assert call(*args, a2.ptr, None, None, None) == fa.FMMH_OK
    hip.synchronize()
    A, P, F = a.download(), p.download(), f.download()
    assert np.array_equal(A, a2.download())
    L = np.longdouble
    # n / 256 + 1 terms a thread, 6 + 3 of the block, 12 within a term; two ranges
    # and their 4 from 16384 bodies on
    bound = (n / 256 + 1 + 9 + 12 + 4) * 2.0 ** -53
    for t in np.unique(np.r_[0:min(nt, 40), max(0, nt - 8):nt]):
        o = np.arange(n) != ids[t]
        d = pos[o].astype(L) - pos[ids[t]].astype(L)
        inv = 1 / np.sqrt((d * d).sum(1) + L(1e-2) * L(1e-2))
        m = mass[o].astype(L)
        term = (m * inv ** 3)[:, None] * d
        assert (np.abs(A[t] - term.sum(0)) <= bound * np.abs(term).sum(0)).all()
        assert abs(P[t] - (m * inv).sum()) <= bound * (m * inv).sum()
        assert abs(F[t] - (m * inv * inv).sum()) <= bound * (m * inv * inv).sum()
    for q in (*bufs, a, p, f, a2):
        q.free()
