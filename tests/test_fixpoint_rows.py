"""The batched Newton solver's row slices at their edges: grids around one slice, one pass of the
workgroup and the two size classes, long rows, isolated vertices, and grids whose matrix does
and does not fit LDS -- the residual in numpy, and the linear solve against a dense one."""
import numpy as np
import pytest


def _star(ND, leaves):
    return ND.SimpleGraph(leaves + 1, np.ones(leaves, np.int64), np.arange(2, leaves + 2))


GRAPHS = [lambda ND: ND.path_graph(2), lambda ND: ND.cycle_graph(63), lambda ND: ND.cycle_graph(64),
          lambda ND: ND.complete_graph(65), lambda ND: _star(ND, 130), lambda ND: ND.barabasi_albert(511, 3, seed=1),
          lambda ND: ND.barabasi_albert(513, 3, seed=2), lambda ND: ND.barabasi_albert(2048, 3, seed=3),
          lambda ND: ND.barabasi_albert(2049, 3, seed=4), lambda ND: ND.barabasi_albert(3500, 4, seed=5),
          lambda ND: ND.barabasi_albert(5120, 2, seed=6), lambda ND: ND.erdos_renyi(600, 30000, seed=7)]


def _residual(g, theta, P, scale, K):
    s, d = g.src - 1, g.dst - 1
    y = K * np.sin(theta[d] - theta[s])
    n = g.nv()
    return (P + np.bincount(s, y, n) - np.bincount(d, y, n)) / scale


@pytest.mark.gpu
def test_newton_slices(ND, dev):
    import torch
    gs = [f(ND) for f in GRAPHS]
    rng = np.random.default_rng(1)
    fs = ND.FixpointSolver(gs)
    P, S, K = [], [], []
    for g in gs:
        p = rng.normal(scale=0.05, size=g.nv())
        P.append(p - p.mean())
        S.append(rng.uniform(0.5, 2.0, g.nv()))
        K.append(rng.uniform(5.0, 15.0, g.ne()))
    up = lambda x: torch.from_numpy(np.concatenate(x)).to(dev)
    for kw in (dict(), dict(inexact=False)):
        th = torch.zeros(int(fs.voff[-1]), dtype=torch.float64, device=dev)
        st = ND.FixpointSolver.stats_to_numpy(fs.solve(th, up(P), up(S), up(K), tol=1e-11, **kw))
        assert (st["retcode"] == 0).all()
        t = th.cpu().numpy()
        for i, g in enumerate(gs):
            r = _residual(g, t[fs.voff[i]:fs.voff[i + 1]], P[i], S[i], K[i])
            # the solver's own residual is below tol; the sums differ by rounding only
            deg = g.degree().max()
            assert np.abs(r).max() <= 1e-11 + 2 * deg * deg * 15.0 * 2.2e-16, i
            assert abs(np.abs(r).max() - st["residual"][i]) <= 2 * deg * deg * 15.0 * 2.2e-16, i
    # L_K theta = P against a dense solve, each up to its mean
    th = torch.zeros(int(fs.voff[-1]), dtype=torch.float64, device=dev)
    st = ND.FixpointSolver.stats_to_numpy(fs.solve(th, up(P), up(S), up(K), tol=1e-12, linearized=True))
    assert (st["retcode"] == 0).all()
    t = th.cpu().numpy()
    for i, g in enumerate(gs):
        n = g.nv()
        if n > 600:
            continue
        L = np.zeros((n, n))
        s, d = g.src - 1, g.dst - 1
        np.add.at(L, (s, s), K[i])
        np.add.at(L, (d, d), K[i])
        np.add.at(L, (s, d), -K[i])
        np.add.at(L, (d, s), -K[i])
        ref = np.linalg.solve(L + 1.0 / n, P[i])
        got = t[fs.voff[i]:fs.voff[i + 1]]
        lam = np.linalg.eigvalsh(L)[1]
        # a residual of at most tol * scale per vertex, over the smallest eigenvalue, and the
        # dense solve's rounding
        bound = (1e-12 * 2.0 * np.sqrt(n) + n * 2.2e-16 * np.abs(L).max() * np.abs(ref).max()) / lam
        assert np.abs((got - got.mean()) - (ref - ref.mean())).max() <= bound, i
