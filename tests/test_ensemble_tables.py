"""Ensembles of lines with two parameters whose edge tables do not fit LDS beside the states,
terms and parameters -- against the oracle's RK4.  With m lines an instance is accepted up to
32 m + 10 n + 12 (chunks of 8 list entries) bytes and takes about 40 m + 8 n with its tables."""
import numpy as np
import pytest

from conftest import oracle_for

LDS = 160 * 1024
GRAPHS = {
    "dense": lambda ND: ND.erdos_renyi(110, 4400, seed=7),
    "sparse": lambda ND: ND.barabasi_albert(1300, 3, seed=8),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(GRAPHS))
def test_static_lines_with_tables_in_memory(ND, dev, name):
    import torch
    g, em = GRAPHS[name](ND), ND.Lib.static_line_edge()
    n, e = g.nv(), g.ne()
    assert 40 * e + 8 * n > LDS
    rng = np.random.default_rng(len(name))
    M, D, P, K = ND.workloads.swing_params(n, e, rng)
    if name == "dense":
        K /= 20.0                                    # about 80 lines per vertex
    p = np.empty(3 * n + 2 * e)
    p[0:3 * n:3], p[1:3 * n:3], p[2:3 * n:3] = M, D, P
    p[3 * n:] = np.stack([K, rng.uniform(0, 0.1, e)], axis=1).reshape(-1)
    u0 = np.empty(2 * n)
    u0[0::2], u0[1::2] = rng.uniform(-1, 1, n), rng.normal(scale=0.5, size=n)
    ens = ND.Ensemble([g, g], ND.Lib.kuramoto_second(), em)     # the second instance at an offset
    u = torch.from_numpy(np.concatenate([u0, u0])).to(dev)
    pd = torch.from_numpy(np.concatenate([p, p])).to(dev)
    st = ND.Ensemble.stats_to_numpy(ens.solve(u, pd, (0.0, 0.1), method=ND.ensemble.RK4, dt=0.005))
    assert (st["retcode"] == 0).all() and (st["naccept"] == 20).all()
    got = u.cpu().numpy().reshape(2, -1)
    assert np.array_equal(got[0], got[1])
    ref = oracle_for(ND.Network(g, ND.Lib.kuramoto_second(), em)).rk4(u0, p, 0.0, 0.005, 20)
    # 80 evaluations, each of rounding error below (terms of the longest row + 20) ulp of a
    # derivative of at most max|P| + deg * K, and a growth over 0.1 time units below e
    deg = g.degree().max()
    tol = 3.0 * 80 * (deg + 20) * 2.2e-16 * 0.005 * (np.abs(P).max() + deg * np.abs(K).max() + 1.0) + 1e-15
    assert np.abs(got[0] - ref).max() <= tol * max(1.0, np.abs(ref).max())
