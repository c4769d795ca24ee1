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


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("n", [70, 2100])
def test_angle_of_a_vertex_without_lines(ND, dev, n, bad):
    # the last vertex has no lines, so its angle enters no equation: a path of the others is solved
    # as it is without that vertex, whatever the angle is
    g = ND.SimpleGraph(n, np.arange(1, n - 1), np.arange(2, n))
    rng = np.random.default_rng(3)
    P = np.r_[rng.normal(0.0, 0.01, n - 1), 0.0]
    P[:-1] -= P[:-1].mean()
    K = rng.uniform(5.0, 10.0, n - 2)
    theta = np.zeros(n)
    ref, st0 = _solve(ND, dev, [g], P, K, theta)
    assert st0["retcode"][0] == 0
    theta[-1] = bad
    th, st = _solve(ND, dev, [g], P, K, theta)
    assert st["retcode"][0] == 0 and st["newton_iters"][0] == st0["newton_iters"][0]
    assert np.array_equal(th[:-1], ref[:-1])
