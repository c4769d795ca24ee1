"""The fused vertex kernel's wave table at its edges: runs of vertices without lines, waves cut
by their vertex count and by their entry count, a vertex with more entries than a window, and a
wave table of full windows -- in both gather modes, against the oracle."""
import numpy as np
import pytest

from conftest import oracle_for, scaled_error


def _star(ND, leaves):
    return ND.SimpleGraph(leaves + 1, np.ones(leaves, np.int64), np.arange(2, leaves + 2))


GRAPHS = {
    "isolated_runs": lambda ND: ND.SimpleGraph(400, [1, 130, 131, 300], [2, 131, 260, 399]),
    "path_1000": lambda ND: ND.path_graph(1000),
    "star_63": lambda ND: _star(ND, 63),
    "star_64": lambda ND: _star(ND, 64),
    "star_65": lambda ND: _star(ND, 65),
    "star_300": lambda ND: _star(ND, 300),
    "er_dense": lambda ND: ND.erdos_renyi(500, 15000, seed=3),
    "ba_150001": lambda ND: ND.barabasi_albert(150_001, 2, seed=4),
}


@pytest.mark.gpu
@pytest.mark.parametrize("vertex", ["swing", "kuramoto"])
@pytest.mark.parametrize("edge", ["kuramoto", "static_line", "diffusion"])
@pytest.mark.parametrize("name", list(GRAPHS))
def test_rhs_wave_table_matches_oracle(ND, dev, name, vertex, edge):
    import torch
    g = GRAPHS[name](ND)
    vm = ND.Lib.kuramoto_second() if vertex == "swing" else ND.Lib.kuramoto_first()
    em = {"kuramoto": ND.Lib.kuramoto_edge, "static_line": ND.Lib.static_line_edge,
          "diffusion": ND.Lib.diffusion_edge}[edge]()
    nw = ND.Network(g, vm, em)
    rng = np.random.default_rng(11)
    u, p = rng.uniform(-3, 3, nw.dim), rng.uniform(0.5, 2.0, nw.pdim)
    on = oracle_for(nw)
    ref, S = on.rhs(u, p, 0.0), on.scale(u, p, 0.0)
    ud, pd = torch.from_numpy(u).to(dev), torch.from_numpy(p).to(dev)
    for mode in (2, 3):
        # every segment on the low path, in the reference order
        nw.tune(gather_mode=mode, hub_degree=1 << 30, big_hub_degree=1 << 30)
        for _ in range(2):
            du = torch.full((nw.dim,), float("nan"), dtype=torch.float64, device=dev)
            nw(du, ud, pd, 0.0)
            assert scaled_error(du.cpu().numpy(), ref, S).max() <= 1e-12
        pd2 = pd * 1.5                               # changed parameters reach the lists
        nw(du, ud, pd2, 0.0)
        ref2, S2 = on.rhs(u, p * 1.5, 0.0), on.scale(u, p * 1.5, 0.0)
        assert scaled_error(du.cpu().numpy(), ref2, S2).max() <= 1e-12
