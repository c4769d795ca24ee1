"""Scratch memory of Network.jvp_multi: taken only where the library uses it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(ND, kind):
    L = ND.Lib
    if kind == "compact":                  # outputs in the compact array, which the plan owns
        return ND.Network(ND.barabasi_albert(1 << 18, 2, seed=1), L.kuramoto_second(), L.kuramoto_edge())
    if kind == "ode":
        return ND.Network(ND.barabasi_albert(30_000, 2, seed=1), L.diffusion_vertex(), L.diffusion_odeedge())
    if kind == "two_edge_batches":
        g = ND.barabasi_albert(60_000, 2, seed=1)
        return ND.Network(g, L.kuramoto_second(), [L.kuramoto_edge() if i % 2 else L.diffusion_edge() for i in range(g.ne())])
    if kind == "near":                     # neighbours have neighbouring numbers
        return ND.Network(ND.path_graph(120_000), L.kuramoto_first(), L.kuramoto_edge())
    return ND.Network(ND.barabasi_albert(60_000, 2, seed=1), L.kuramoto_second(), L.kuramoto_edge())


@pytest.mark.parametrize("kind,used", [("compact", False), ("ode", False), ("two_edge_batches", False), ("near", False),
                                       ("random", True)])
def test_scratch_only_where_it_is_read(ND, dev, kind, used):
    import torch
    nw = _net(ND, kind)
    rng = np.random.default_rng(1)
    d = lambda x: torch.from_numpy(x).to(dev)
    u, p, V = d(rng.normal(size=nw.dim)), d(rng.uniform(0.5, 2.0, nw.pdim)), d(rng.normal(size=(8, nw.dim)))
    du, jv, du2, jv2 = torch.empty_like(u), torch.empty_like(V), torch.empty_like(u), torch.empty_like(V)
    lib = ND._abi.lib()
    assert nw.dim >= 100_000
    assert lib.nd_rhs_jvp_multi_scratch(nw.plan, 8) == (8 * nw.dim if used else 0)
    assert lib.nd_rhs_jvp_multi_scratch(nw.plan, 4) == lib.nd_rhs_jvp_multi_scratch(nw.plan, 9) == 0
    nw.jvp_multi(du, jv, u, V, p)          # buffers of the plan's own are made here
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    nw.jvp_multi(du, jv, u, V, p)
    extra = torch.cuda.max_memory_allocated() - before
    assert extra >= 64 * nw.dim if used else extra == 0
    ND._abi.check(lib.nd_rhs_jvp_multi(nw.plan, du2.data_ptr(), jv2.data_ptr(), u.data_ptr(), V.data_ptr(), 8, p.data_ptr(),
                                       0.0, nw.dim, nw.dim, nw.pdim, torch.cuda.current_stream(dev).cuda_stream))
    assert torch.equal(du, du2) and torch.equal(jv, jv2)


def test_null_plan_needs_none(ND, dev):
    assert ND._abi.lib().nd_rhs_jvp_multi_scratch(None, 8) == 0
