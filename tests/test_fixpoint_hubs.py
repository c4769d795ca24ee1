"""Long rows of the batched Newton solver, which a whole wave evaluates: hubs around one and two
columns of 64 entries, several hubs per wave, hubs in both size classes and with their columns in
and outside LDS -- the residual in numpy, and the same bits where other vertices make the rows
sliced."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _hubs(ND, hubs, leaves, ring, alone=0):
    """A ring of `ring` vertices, `hubs` of them joined to `leaves` vertices of their own."""
    e = [(i, i + 1) for i in range(1, ring)] + [(1, ring)]
    n = ring
    for h in range(hubs):
        e += [(1 + h * (ring // hubs), n + 1 + j) for j in range(leaves)]
        n += leaves
    e = np.array(sorted(e))
    return ND.SimpleGraph(n + alone, e[:, 0], e[:, 1])


CASES = [(1, 62, 10, 0), (1, 63, 10, 3), (1, 126, 5, 0), (1, 127, 700, 0), (3, 200, 30, 0), (9, 64, 90, 1), (20, 90, 40, 0),
         (1, 1900, 60, 0), (1, 5000, 100, 0), (30, 100, 2000, 0), (2, 1200, 2600, 5)]


def _solve(ND, dev, gs, P, S, K, **kw):
    import torch
    up = lambda x: torch.from_numpy(np.concatenate(x)).to(dev)
    fs = ND.FixpointSolver(gs)
    th = torch.zeros(int(fs.voff[-1]), dtype=torch.float64, device=dev)
    st = ND.FixpointSolver.stats_to_numpy(fs.solve(th, up(P), up(S), up(K), **kw))
    t = th.cpu().numpy()
    return [t[fs.voff[i]:fs.voff[i + 1]] for i in range(len(gs))], st


@pytest.mark.parametrize("kw", [dict(), dict(inexact=False), dict(linearized=True)], ids=["inexact", "exact", "linearized"])
def test_hubs(ND, dev, kw):
    gs = [_hubs(ND, *c) for c in CASES]
    rng = np.random.default_rng(2)
    P, S, K = [], [], []
    for c, g in zip(CASES, gs):
        p = rng.normal(scale=0.01, size=g.nv())
        m = g.nv() - c[3]                                # the vertices alone need no injection
        p[m:] = 0.0
        p[:m] -= p[:m].mean()
        P.append(p)
        S.append(rng.uniform(0.5, 2.0, g.nv()))
        K.append(rng.uniform(5.0, 15.0, g.ne()))
    th, st = _solve(ND, dev, gs, P, S, K, tol=1e-11, **kw)
    # the long ring's last system is beyond what 20000 exact CG iterations reach, with its rows in
    # slices as well
    ok = st["retcode"] == 0
    assert ok[:-1].all() and (ok[-1] or "inexact" in kw)
    for i, g in enumerate(gs):
        if not ok[i]:
            continue
        s, d, n = g.src - 1, g.dst - 1, g.nv()
        D = th[i][d] - th[i][s]
        y = K[i] * (D if kw.get("linearized") else np.sin(D))
        r = (P[i] + np.bincount(s, y, n) - np.bincount(d, y, n)) / S[i]
        # the solver's own residual is below tol; the sums differ by rounding only
        deg = g.degree().max()
        slack = 2 * deg * deg * 15.0 * 2.2e-16
        assert np.abs(r).max() <= 1e-11 + slack, i
        assert abs(np.abs(r).max() - st["residual"][i]) <= slack, i
    # each grid by itself, whose columns then have the whole LDS: the same bits
    for i in (4, 6, 7, 9):
        one, st1 = _solve(ND, dev, [gs[i]], [P[i]], [S[i]], [K[i]], tol=1e-11, **kw)
        assert np.array_equal(one[0], th[i]) and st1["cg_iters"][0] == st["cg_iters"][i]
