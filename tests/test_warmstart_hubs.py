"""Rows of the warm-start network's graph that are longer than the 96 entries a wave sums beside
those of its tile's other nodes: lengths around 96 and the 32 and 64 of the long rows' steps,
several in a tile and one in a tile by itself, forward and backward against float64."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mpnn_ref  # noqa: E402

LENGTHS = (63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 161, 1000)


def _graph(n, seed):
    """A ring, LENGTHS[i] lines at node 18 + i and 2000 at node 101 where there are as many nodes."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    e = {(i, (i + 1) % n) for i in range(n)}
    for i, k in enumerate(LENGTHS):
        e |= {(18 + i, j) for j in range(40, 40 + k - 2)}          # two more on the ring
    if n > 2200:
        e |= {(101, j) for j in range(200, 2200)}
    s, d = np.array(sorted(e)).T
    w = rng.uniform(1.0, 2.0, len(s))
    M = sp.csr_matrix((np.r_[w, w], (np.r_[s, d], np.r_[d, s])), shape=(n, n))
    A = sp.csr_matrix(sp.diags(1.0 / np.asarray(M.sum(axis=1)).ravel()) @ M)
    A.sort_indices()
    return A


@pytest.mark.gpu
@pytest.mark.parametrize("n,nfeat", [(1100, 8), (1101, 5), (2500, 8), (40_000, 8)])
def test_long_rows(ND, dev, n, nfeat):
    # a row of 2000 entries: 96 + 1904 / 4 + 2 sums in a row, and 128 products, each rounded to 6e-8:
    # 4e-5 a layer at the very worst, 2e-4 over five.  Float32 also decides a few of the n * 320
    # rectifiers the other way (sums within 1e-6 of zero), each of which moves the gradients by about
    # 1 / n: compared in norm with twice the forward bound
    import torch
    A = _graph(n, n)
    rng = np.random.default_rng(n)
    params = rng.normal(0, 0.15, nfeat * 64 + 64 + 4 * (64 * 128 + 64) + 65).astype(np.float32)
    X, y = rng.normal(size=(n, nfeat)).astype(np.float32), rng.normal(size=n).astype(np.float32)
    At = A.T.tocsr()
    At.sort_indices()
    assert np.array_equal(At.indices, A.indices)
    d = lambda x, dt: torch.from_numpy(np.ascontiguousarray(x, dt)).to(dev)
    rp, nb, af, ab = d(A.indptr, np.int32), d(A.indices, np.int32), d(A.data, np.float32), d(At.data, np.float32)
    p, Xd, yd = d(params, np.float32), d(X, np.float32), d(y, np.float32)
    L = ND._abi.lib()
    work = torch.full((int(L.nd_mp_workspace_floats(n)),), float("nan"), dtype=torch.float32, device=dev)
    out, g = torch.full((n,), float("nan"), dtype=torch.float32, device=dev), torch.full_like(p, float("nan"))
    lp = torch.zeros(n // 4 + 2, dtype=torch.float32, device=dev)
    s = torch.cuda.current_stream(dev).cuda_stream
    ND._abi.check(L.nd_mp_forward(n, rp.data_ptr(), nb.data_ptr(), af.data_ptr(), Xd.data_ptr(), nfeat, p.data_ptr(),
                                  work.data_ptr(), out.data_ptr(), s))
    ND._abi.check(L.nd_mp_backward(n, rp.data_ptr(), nb.data_ptr(), ab.data_ptr(), Xd.data_ptr(), nfeat, p.data_ptr(),
                                   yd.data_ptr(), work.data_ptr(), g.data_ptr(), lp.data_ptr(), s))
    ref, _ = mpnn_ref.forward(params, X, A)
    loss, gref = mpnn_ref.loss_and_grad(params, X, A, y)
    got, gg = out.cpu().numpy(), g.cpu().numpy()
    assert np.abs(got - ref).max() <= 2e-4 * np.abs(ref).max()
    assert np.linalg.norm(gg - gref) <= 4e-4 * np.linalg.norm(gref)
    assert abs(lp.sum().item() / n - loss) <= 2e-4 * loss
