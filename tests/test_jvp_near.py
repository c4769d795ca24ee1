"""Jacobian-vector products of networks whose numbering puts neighbours together, which take a
thread per vertex: sixteen copies of a network side by side give sixteen times its results, bit
for bit, in every edge form, with rows on either side of a workgroup's length and vertices
without lines."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
COPIES = 16


def _part(ND):
    """A path with chords, centres with 3, 64, 65 and 300 leaves next to them, and vertices alone:
    1501 vertices, about 2 entries a row."""
    e, n = [(i, i + 1) for i in range(1, 900)] + [(i, i + 5) for i in range(1, 890, 7)], 900
    for k in (3, 64, 65, 300):
        centre = n + k // 2                       # leaves on both sides: rows of both directions
        e += [(min(centre, x), max(centre, x)) for x in range(n + 1, n + k + 2) if x != centre]
        n += k + 1
    e = np.array(sorted(e))
    return 1501, e[:, 0], e[:, 1]


def _models(ND, kind, n, m):
    L = ND.Lib
    one = {"kuramoto": (L.kuramoto_first(), L.kuramoto_edge()), "swing": (L.kuramoto_second(), L.kuramoto_edge()),
           "lines": ([L.kuramoto_second() if i % 3 else L.load_vertex() for i in range(n)], L.static_line_edge()),
           "diffusion": (L.diffusion_vertex(), L.diffusion_edge()), "fiducial": (L.diffusion_vertex(), L.diffusion_edge_fid()),
           "ode": (L.diffusion_vertex(), L.diffusion_odeedge()), "lag": (L.kuramoto_second(), L.ode_lag_edge("anti")),
           "mixed": (L.kuramoto_second(), [L.kuramoto_edge() if i % 2 else L.diffusion_edge() for i in range(m)])}
    return one[kind]


def _net(ND, kind, copies):
    n, s, d = _part(ND)
    S = np.concatenate([s + c * n for c in range(copies)])
    D = np.concatenate([d + c * n for c in range(copies)])
    vm, em = _models(ND, kind, n, len(s))
    vm = vm * copies if isinstance(vm, list) else vm
    em = em * copies if isinstance(em, list) else em
    return ND.Network(ND.SimpleGraph(copies * n, S, D), vm, em), n, len(s)


def _places(nw, n, m, copy):
    """States and parameters of one copy, in the order of the single network's."""
    v, e = nw.ranges()

    def of(r, col, lo, cnt):
        return np.concatenate([np.arange(a - 1, b) for a, b in r[lo:lo + cnt, col]])
    st = np.concatenate([of(v, 0, copy * n, n), of(e, 0, copy * m, m)])
    par = np.concatenate([of(v, 2, copy * n, n), of(e, 3, copy * m, m)])
    return st, par


@pytest.mark.parametrize("gather", [2, 3])
@pytest.mark.parametrize("kind", ["kuramoto", "swing", "lines", "diffusion", "fiducial", "ode", "lag", "mixed"])
def test_copies_side_by_side(ND, dev, kind, gather):
    import torch
    one, n, m = _net(ND, kind, 1)
    many, _, _ = _net(ND, kind, COPIES)
    rng = np.random.default_rng(7)
    u1, p1, V1 = rng.normal(size=one.dim), rng.uniform(0.5, 2.0, one.pdim), rng.normal(size=(8, one.dim))
    s1, q1 = _places(one, n, m, 0)
    u, p, V = np.empty(many.dim), np.empty(many.pdim), np.empty((8, many.dim))
    places = [_places(many, n, m, c) for c in range(COPIES)]
    for st, par in places:
        u[st], p[par], V[:, st] = u1[s1], p1[q1], V1[:, s1]
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)
    for nw in (one, many):
        nw.tune(gather_mode=gather)
    ud, pd, Vd, u1d, p1d, V1d = d(u), d(p), d(V), d(u1), d(p1), d(V1)
    for k in (1, 2, 4, 5, 8):
        du, jv = torch.full_like(ud, np.nan), torch.full_like(Vd[:k], np.nan)
        du1, jv1 = torch.full_like(u1d, np.nan), torch.full_like(V1d[:k], np.nan)
        one.jvp_multi(du1, jv1, u1d, V1d[:k].contiguous(), p1d)
        many.jvp_multi(du, jv, ud, Vd[:k].contiguous(), pd)
        du, jv, du1, jv1 = (x.cpu().numpy() for x in (du, jv, du1, jv1))
        assert np.isfinite(du).all() and np.isfinite(jv).all()
        for st, _ in places:
            assert np.array_equal(du[st], du1[s1]) and np.array_equal(jv[:, st], jv1[:, s1])
