"""Jacobian-vector products over rows of every kind: shorter and longer than the lanes of a
vertex, on either side of the length from which a row gets a workgroup of its own, longer than
a workgroup, and none at all; one tangent against the closed form, several against one at a
time."""
import numpy as np
import pytest
from conftest import oracle_for, scaled_error

RTOL = 1e-12
pytestmark = pytest.mark.gpu


def _rows_graph(ND):
    """Centres with 1, 7, 8, 9, 63, 64, 65, 256, 257 and 600 leaves, then two vertices alone."""
    src, dst, n = [], [], 0
    for k in (1, 7, 8, 9, 63, 64, 65, 256, 257, 600):
        centre = n + 1
        for leaf in range(centre + 1, centre + 1 + k):
            # alternate directions: rows hold source and destination entries
            a, b = (centre, leaf) if leaf % 2 else (leaf, centre)
            src.append(min(a, b))
            dst.append(max(a, b))
        n += k + 1
    return ND.SimpleGraph(n + 2, np.array(src), np.array(dst))


@pytest.mark.parametrize("kind", ["kuramoto", "swing"])
@pytest.mark.parametrize("gather", [2, 3])
def test_rows_of_every_length(ND, dev, kind, gather):
    # RTOL: the bound of the other closed-form checks (sums of up to 600 terms in row order)
    import torch
    from test_oracle import kuramoto_jvp_closed_form, swing_jvp_closed_form
    rng = np.random.default_rng(5)
    g = _rows_graph(ND)
    n, m = g.nv(), g.ne()
    K = rng.uniform(0.5, 2.0, m)
    if kind == "kuramoto":
        nw, p = ND.Network(g, ND.Lib.kuramoto_first(), ND.Lib.kuramoto_edge()), np.r_[rng.normal(size=n), K]
    else:
        nw = ND.Network(g, ND.Lib.kuramoto_second(), ND.Lib.kuramoto_edge())
        M, D = rng.uniform(1, 5, n), rng.uniform(0.1, 1, n)
        p = np.r_[np.stack([M, D, rng.normal(size=n)], 1).ravel(), K]
    nw.tune(gather_mode=gather)
    u, V = rng.normal(size=nw.dim), rng.normal(size=(8, nw.dim))
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    nan = lambda *s: torch.full(s, float("nan"), dtype=torch.float64, device=dev)
    ud, pd, Vd = d(u), d(p), d(V)
    du, jv = nan(nw.dim), nan(8, nw.dim)
    for j in range(8):
        nw.jvp(du, jv[j], ud, Vd[j], pd, 0.0)
    for j in (0, 7):
        ref, S = kuramoto_jvp_closed_form(g, u, K, V[j]) if kind == "kuramoto" else \
            swing_jvp_closed_form(g, u, M, D, K, V[j])
        assert scaled_error(jv[j].cpu().numpy(), ref, S).max() <= RTOL
    on = oracle_for(nw)
    assert scaled_error(du.cpu().numpy(), on.rhs(u, p), on.scale(u, p)).max() <= RTOL
    for k in (1, 2, 4, 5, 8):
        duk, jvk = nan(nw.dim), nan(8, nw.dim)
        nw.jvp_multi(duk, jvk[:k], ud, Vd[:k], pd, 0.0)
        assert torch.equal(duk, du) and torch.equal(jvk[:k], jv[:k]) and bool(jvk[k:].isnan().all())
        # with scratch memory: the tangents of more than four columns row by row; a scratch too short
        # or not 16-byte aligned is not used
        work = nan(8 * nw.dim + 1)
        for first, length in ((0, 8 * nw.dim), (1, 8 * nw.dim), (0, 8 * nw.dim - 1)):
            duk, jvk = nan(nw.dim), nan(8, nw.dim)
            ND._abi.check(ND._abi.lib().nd_rhs_jvp_multi_work(
                nw.plan, duk.data_ptr(), jvk.data_ptr(), ud.data_ptr(), Vd.data_ptr(), k, pd.data_ptr(), 0.0,
                work.data_ptr() + 8 * first, length, nw.dim, nw.dim, nw.pdim, torch.cuda.current_stream(dev).cuda_stream))
            assert torch.equal(duk, du) and torch.equal(jvk[:k], jv[:k]) and bool(jvk[k:].isnan().all())
