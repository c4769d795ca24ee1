"""The ensemble kernel's row layout at its edges: rows of odd length, empty rows, rows at and
above the length one thread sums by itself, edge counts that are no multiple of the edge
batch, and an instance whose tables do not fit LDS -- all against the oracle's RK4."""
import numpy as np
import pytest

from conftest import oracle_for


def _star(ND, leaves, extra=0):
    return ND.SimpleGraph(leaves + 1 + extra, np.ones(leaves, np.int64), np.arange(2, leaves + 2))


GRAPHS = {
    "one_edge": lambda ND: ND.path_graph(2),
    "two_edges": lambda ND: ND.path_graph(3),
    "five_edges_isolated_vertices": lambda ND: ND.SimpleGraph(70, [1, 1, 2, 3, 64], [2, 3, 3, 4, 65]),
    "star_16": lambda ND: _star(ND, 16),
    "star_17": lambda ND: _star(ND, 17, extra=3),
    "star_40": lambda ND: _star(ND, 40),
    "star_301": lambda ND: _star(ND, 301),
    "complete_9": lambda ND: ND.complete_graph(9),
    "complete_18": lambda ND: ND.complete_graph(18),
    "ba_1025": lambda ND: ND.barabasi_albert(1025, 2, seed=5),
    "ba_2000": lambda ND: ND.barabasi_albert(2000, 2, seed=6),
    "tables_in_memory": lambda ND: ND.erdos_renyi(110, 5400, seed=7),
}


@pytest.mark.gpu
@pytest.mark.parametrize("line", [False, True], ids=["kuramoto_edge", "static_line"])
@pytest.mark.parametrize("name", list(GRAPHS))
def test_ensemble_rows_match_oracle(ND, dev, name, line):
    import torch
    if line and name in ("ba_2000", "tables_in_memory"):
        pytest.skip("two parameters per edge: above the kernel's size limit")
    g = GRAPHS[name](ND)
    rng = np.random.default_rng(len(name))
    n, e = g.nv(), g.ne()
    em = ND.Lib.static_line_edge() if line else ND.Lib.kuramoto_edge()
    M, D, P, K = ND.workloads.swing_params(n, e, rng)
    if name == "tables_in_memory":
        K /= 20.0                                    # about 100 lines per vertex
    p = np.empty(3 * n + e * (2 if line else 1))
    p[0:3 * n:3], p[1:3 * n:3], p[2:3 * n:3] = M, D, P
    p[3 * n:] = np.stack([K, rng.uniform(0, 0.1, e)], axis=1).reshape(-1) if line else K
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
