"""The ensemble's kernels by workgroup size: two edges at a time against four where a small
workgroup has at most two per thread, and RK4's registers for few and for many instances.  RK4
gives the same bits in every shape; Tsit5's error norm is summed in another order, so its
solutions agree to the tolerance."""
import numpy as np
import pytest

from conftest import oracle_for

pytestmark = pytest.mark.gpu
SHAPES = [(64, 1), (64, 2), (64, 4), (128, 1), (128, 2), (192, 1), (256, 1), (256, 2), (320, 1), (512, 1), (512, 2), (512, 3),
          (1024, 1)]


def _problem(ND, n, m, swing, seed):
    """n vertices and m edges: a path, then random chords."""
    rng = np.random.default_rng(seed)
    e = {(i, i + 1) for i in range(1, min(n, m + 1))}
    while len(e) < m:
        a, b = rng.integers(1, n + 1, 2)
        if a != b:
            e.add((min(a, b), max(a, b)))
    e = np.array(sorted(e))
    g = ND.SimpleGraph(n, e[:, 0], e[:, 1])
    M, D, P, K = ND.workloads.swing_params(n, m, rng)
    K /= 4.0
    if swing:
        u = np.empty(2 * n)
        u[0::2], u[1::2] = rng.uniform(-1, 1, n), rng.normal(scale=0.5, size=n)
        return g, u, np.r_[np.stack([M, D, P], axis=1).ravel(), K]
    return g, rng.uniform(-1, 1, n), np.r_[P, K]


def _solve(ND, dev, g, u, p, copies, shape, swing, **kw):
    import torch
    L = ND.Lib
    ens = ND.Ensemble([g] * copies, L.kuramoto_second() if swing else L.kuramoto_first(), L.kuramoto_edge())
    ens.set_classes([shape])
    ud, pd = torch.from_numpy(np.tile(u, copies)).to(dev), torch.from_numpy(np.tile(p, copies)).to(dev)
    if kw.pop("limits", False):
        kw["line_limit"] = torch.full((copies * g.ne(),), 1e9, dtype=torch.float64, device=dev)
    st = ND.Ensemble.stats_to_numpy(ens.solve(ud, pd, (0.0, 0.2), **kw))
    assert (st["retcode"] == 0).all()
    out = ud.cpu().numpy().reshape(copies, -1)
    assert (out == out[0]).all()
    return out[0]


@pytest.mark.parametrize("swing", [True, False], ids=["swing", "kuramoto"])
@pytest.mark.parametrize("n,m", [(60, 1), (60, 127), (61, 128), (62, 129), (60, 255), (60, 256), (60, 257), (63, 512), (63, 513)])
def test_shapes(ND, dev, n, m, swing):
    g, u, p = _problem(ND, n, m, swing, n + m)
    fits = [s for s in SHAPES if s[0] * s[1] >= n]
    rk = dict(method=ND.ensemble.RK4, dt=0.01)
    ref = _solve(ND, dev, g, u, p, 2, fits[0], swing, **rk)
    for s in fits[1:]:
        assert np.array_equal(_solve(ND, dev, g, u, p, 2, s, swing, **rk), ref)
    vm = ND.Lib.kuramoto_second() if swing else ND.Lib.kuramoto_first()
    on = oracle_for(ND.Network(g, vm, ND.Lib.kuramoto_edge())).rk4(u, p, 0.0, 0.01, 20)
    # 80 evaluations, each of rounding error below (a row's terms + 20) ulp of a derivative of at most
    # max|P| + deg * K, and a growth over 0.2 time units below e
    deg = g.degree().max()
    tol = 3.0 * 80 * (deg + 20) * 2.2e-16 * 0.01 * (5.0 + deg * 2.5) + 1e-15
    assert np.abs(ref - on).max() <= tol * max(1.0, np.abs(on).max())
    for kw in (dict(), dict(limits=True)):
        ts = [_solve(ND, dev, g, u, p, 2, s, swing, **kw) for s in fits]
        for x in ts[1:]:
            # steps that differ in the last bits: the difference is that of the roundings, far below
            # the error of the method at 1e-8
            assert np.abs(x - ts[0]).max() <= 1e-10 * max(1.0, np.abs(ts[0]).max())


@pytest.mark.parametrize("swing", [True, False], ids=["swing", "kuramoto"])
@pytest.mark.parametrize("shape,copies", [((64, 1), 3100), ((64, 2), 3100), ((128, 2), 1600), ((256, 1), 800), ((512, 1), 300),
                                          ((512, 2), 300)])
def test_many_instances(ND, dev, shape, copies, swing):
    g, u, p = _problem(ND, 50, 90, swing, 7)
    rk = dict(method=ND.ensemble.RK4, dt=0.01)
    few = _solve(ND, dev, g, u, p, 2, shape, swing, **rk)
    assert np.array_equal(_solve(ND, dev, g, u, p, copies, shape, swing, **rk), few)
