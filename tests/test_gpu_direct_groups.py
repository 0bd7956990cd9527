"""GPU test of the direct sum's two launch shapes (single targets; groups of
four at the larger sizes): last groups that are not full, ranges that end
inside a stride of 256 sources, targets that repeat or share a stride with
others, the first and the last body, and ids out of range (NaN sums for them,
their group's other targets as they are)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def direct_noalloc(fa, hip, pos, mass, ids, softening):
    nt = len(ids)
    dp, dm = hip.DeviceArray.from_host(pos), hip.DeviceArray.from_host(mass)
    di = hip.DeviceArray.from_host(np.ascontiguousarray(ids, np.uint32))
    a, p, f = hip.DeviceArray((nt, 3)), hip.DeviceArray((nt,)), hip.DeviceArray((nt,))
    rc = fa.lib().fmmh_direct_sampled_noalloc(len(mass), dp.ptr, dm.ptr, float(softening), nt,
                                              di.ptr, a.ptr, p.ptr, f.ptr, None)
    assert rc == fa.FMMH_OK, rc
    hip.synchronize()
    out = a.download(), p.download(), f.download()
    for q in (dp, dm, di, a, p, f):
        q.free()
    return out


@pytest.mark.parametrize("n,nt,soft", [(1, 3, 1e-3), (2, 1, 0.0), (255, 3069, 0.0),
                                       (513, 3100, 1e-2), (8193, 7, 0.0), (70001, 1002, 0.0),
                                       (70001, 381, 1e-3)])
def test_direct_edges_against_extended_precision(n, nt, soft):
    import fmms_amd as fa
    from fmms_amd import hip

    print(f"[direct] n={n} nt={nt} soft={soft}", flush=True)
    rng = np.random.default_rng(n + nt)
    pos, mass = rng.standard_normal((n, 3)), rng.uniform(0.5, 1.5, n)
    ids = rng.integers(0, n, nt).astype(np.uint32)
    ids[0], ids[-1] = 0, n - 1
    if nt > 300:  # one stride with several targets, a repeated target
        ids[1:9] = min(n - 1, 300) - np.array([0, 1, 2, 3, 3, 2, 1, 0])
        ids[20], ids[21] = n, 0xFFFFFFFF  # out of range
    a, p, f = direct_noalloc(fa, hip, pos, mass, ids, soft)
    sel = np.unique(np.r_[0:min(nt, 24), max(0, nt - 6):nt])
    L = np.longdouble
    # Roundings of a sum: at most n / 256 + 1 terms a thread, 6 + 3 of the block,
    # 32 + 3 of the ranges, and 12 within a term; of the terms' absolute sum.
    bound = (n / 256 + 1 + 44 + 12) * 2.0 ** -53
    for t in sel:
        if ids[t] >= n:
            assert np.isnan(a[t]).all() and np.isnan(p[t]) and np.isnan(f[t])
            continue
        o = np.arange(n) != ids[t]
        d = pos[o].astype(L) - pos[ids[t]].astype(L)
        inv = 1 / np.sqrt((d * d).sum(1) + L(soft) * L(soft))
        m = mass[o].astype(L)
        term = (m * inv ** 3)[:, None] * d
        assert (np.abs(a[t] - term.sum(0)) <= bound * np.abs(term).sum(0)).all()
        assert abs(p[t] - (m * inv).sum()) <= bound * (m * inv).sum()
        assert abs(f[t] - (m * inv * inv).sum()) <= bound * (m * inv * inv).sum()
