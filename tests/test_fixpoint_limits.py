"""The fixpoint solver at the limits of its arithmetic."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(ND, dev, graphs, P, K, theta=None, **kw):
    import torch
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x, np.float64)).to(dev)
    th = d(np.zeros(len(P)) if theta is None else theta)
    S = ND.FixpointSolver(graphs)
    st = S.stats_to_numpy(S.solve(th, d(P), d(np.ones(len(P))), d(K), **kw))
    return th.cpu().numpy(), st


@pytest.mark.parametrize("n", [3, 2100])          # the two size classes
def test_weights_that_sum_past_the_largest_double(ND, dev, n):
    # vertex 1 joins two lines of 1e308: its Jacobi diagonal is infinite and its quotients are 0;
    # the other two are one Newton step from their fixpoint theta = P / K
    g = ND.SimpleGraph(n, [1, 1], [2, 3])
    P = np.zeros(n)
    P[1], P[2] = 1e100, -1e100
    th, st = _solve(ND, dev, [g], P, [1e308, 1e308], tol=1e90)
    assert st["retcode"][0] == 0 and st["newton_iters"][0] == 1
    assert np.isfinite(th).all()
    np.testing.assert_allclose(th[1:3] - th[0], [1e-208, -1e-208], rtol=1e-12)
