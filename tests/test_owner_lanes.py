"""The right-hand side of a network with more vertex outputs than an owner lane can share an
entry with (2^25): the lanes lie in an array of their own there.  Compared with the model
written out in float64."""
import pytest


@pytest.mark.gpu
@pytest.mark.timeout(300)
def test_more_outputs_than_an_entry_holds_beside_the_lane(ND, dev):
    import torch
    n = 2**25 + 67
    nw = ND.Network(ND.path_graph(n), ND.Lib.kuramoto_first(), ND.Lib.kuramoto_edge())
    gen = torch.Generator(device=dev).manual_seed(3)
    u = torch.rand(n, generator=gen, device=dev, dtype=torch.float64) * 2 - 1
    om = torch.rand(n, generator=gen, device=dev, dtype=torch.float64) * 2 - 1
    K = torch.rand(n - 1, generator=gen, device=dev, dtype=torch.float64) + 0.5
    assert nw.dim == n and nw.pdim == 2 * n - 1
    p = torch.cat([om, K])
    du = torch.empty_like(u)
    flow = K * torch.sin(u[:-1] - u[1:])          # from vertex i to i + 1
    ref = om.clone()
    ref[1:] += flow
    ref[:-1] -= flow
    # two flows of at most 1.5, each within 2 ulp of its sine and of its product, and two sums
    # of magnitude below 4: below 32 eps in all
    for _ in range(2):                            # the second call reads the parameters' copy
        du.fill_(float("nan"))
        nw(du, u, p, 0.0)
        assert float((du - ref).abs().max()) <= 32 * 2.3e-16
