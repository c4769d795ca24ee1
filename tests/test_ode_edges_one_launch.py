"""ODE edges evaluated in the launch of the vertices that they feed: edge counts around a
workgroup's 256, one and several vertex batches, every wrapper."""
import numpy as np
import pytest

from conftest import oracle_for, scaled_error

RTOL = 1e-12
pytestmark = pytest.mark.gpu


def _network(ND, ne, wrapper, batches, seed):
    L, rng = ND.Lib, np.random.default_rng(seed)
    n = ne + 1 - ne // 4                      # a path and ne // 4 chords
    src = np.r_[np.arange(1, n), np.arange(1, ne // 4 + 1)]
    dst = np.r_[np.arange(2, n + 1), np.arange(1, ne // 4 + 1) + 2]
    g = ND.SimpleGraph(n, src, dst)
    kinds = [L.kuramoto_second(), L.diffusion_vertex(), L.kuramoto_first()]
    vm = [kinds[i % batches] for i in range(n)]
    em = L.diffusion_odeedge() if wrapper == "fiducial" else L.ode_lag_edge(wrapper)
    nw = ND.Network(g, vm, em)
    return nw, rng.normal(size=nw.dim), rng.uniform(0.5, 2.0, nw.pdim)


@pytest.mark.parametrize("ne,wrapper,batches", [(3, "anti", 1), (255, "anti", 1), (256, "sym", 2), (257, "fiducial", 3),
                                                (1025, "fiducial", 1), (300, "directed", 2)])
def test_rhs_and_rk4_match_oracle(ND, dev, ne, wrapper, batches):
    # an evaluation within 1e-12 of the terms' magnitudes (the bound of the other RHS checks); five
    # steps of 0.01 form 20 of them, each weighted by at most the step: 5 * 0.01 * 1e-12 of
    # magnitudes below 100 in all, held to 1e-11
    import torch
    nw, u, p = _network(ND, ne, wrapper, batches, seed=ne)
    on = oracle_for(nw)
    ref, S = on.rhs(u, p), on.scale(u, p)
    end = on.rk4(u, p, 0.0, 0.01, 5)
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    for mode in (2, 3):
        nw.tune(gather_mode=mode)
        du = torch.full((nw.dim,), float("nan"), dtype=torch.float64, device=dev)
        nw(du, d(u), d(p), 0.0)
        assert scaled_error(du.cpu().numpy(), ref, S).max() <= RTOL
        x = d(u)
        nw.rk4(x, d(p), 0.0, 0.01, 5)
        np.testing.assert_allclose(x.cpu().numpy(), end, rtol=1e-11, atol=1e-11)
