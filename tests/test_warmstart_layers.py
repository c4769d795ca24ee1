"""The warm-start network's layer kernels where a tile is not full: node counts around the
16 nodes of a wave and the 64 of a workgroup, a row longer than all others, nodes without
neighbours, feature counts on either side of the input layer's own width, and an input that
is not 16-byte aligned; many copies of one graph against the graph itself, for the workgroup
shapes that larger batches take and rows past a 32-bit byte offset."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mpnn_ref  # noqa: E402


def _problem(n, nfeat):
    """Random symmetric pattern, node 0 joined to every other, the last two nodes without
    neighbours.  The inputs are redrawn until no sum before a ReLU lies within 4e-6 of zero
    (an FP32 sum of 200 terms of order 0.1 to 1 errs by less), so that both sides take the
    same branch everywhere."""
    import scipy.sparse as sp
    rng = np.random.default_rng(100 * n + nfeat)
    M = np.zeros((n, n))
    last = n - 2
    for i in range(1, last):
        M[0, i] = rng.uniform(1, 2)
        for j in rng.choice(last, min(3, last), replace=False):
            if i != j:
                M[i, j] = rng.uniform(1, 2)
    M = np.maximum(M, M.T)
    A = sp.csr_matrix(M / np.maximum(M.sum(axis=1, keepdims=True), 1e-30))
    A.sort_indices()
    while True:
        params = rng.normal(0, 0.15, nfeat * 64 + 64 + 4 * (64 * 128 + 64) + 65).astype(np.float32)
        X = (rng.normal(size=(n, nfeat)) * np.sqrt(8 / nfeat)).astype(np.float32)
        P = mpnn_ref.unpack(params, nfeat)
        _, Hs = mpnn_ref.forward(params, X, A)
        sums = [X.astype(np.float64) @ P["W_in"] + P["b_in"]]
        for l in range(4):
            Y = Hs[l] @ P[f"WU{l}"]
            sums.append(A @ Y[:, :64] + Y[:, 64:] + P[f"b{l}"])
        if min(np.abs(z).min() for z in sums) > 4e-6:
            return A, params, X, rng.normal(size=n).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("n,nfeat,offset", [(1, 8, 0), (2, 8, 0), (15, 8, 0), (17, 8, 1), (63, 8, 0), (64, 5, 0), (65, 8, 0),
                                            (129, 100, 0), (511, 8, 0), (513, 8, 0)])
def test_layers_at_tile_edges(ND, dev, n, nfeat, offset):
    # forward: 5 layers of at most 128 products plus a row's entries, each product and sum
    # rounded to 6e-8: 5 * 200 * 6e-8 = 6e-5 relative at the very worst, 2e-4 with the head;
    # gradients pass through as many layers again and are compared in norm
    import torch
    A, params, X, y = _problem(n, nfeat)
    D = A.toarray()
    rows = np.repeat(np.arange(n), np.diff(A.indptr))
    d = lambda x, dt: torch.from_numpy(np.ascontiguousarray(x, dt)).to(dev)
    rp, nb = d(A.indptr, np.int32), d(A.indices if A.nnz else [0], np.int32)
    af, ab = d(A.data if A.nnz else [0], np.float32), d(D.T[rows, A.indices] if A.nnz else [0], np.float32)
    p, yd = d(params, np.float32), d(y, np.float32)
    Xd = torch.empty(n * nfeat + offset, dtype=torch.float32, device=dev)[offset:]
    Xd.copy_(d(X, np.float32).reshape(-1))
    L = ND._abi.lib()
    work = torch.full((int(L.nd_mp_workspace_floats(n)),), float("nan"), dtype=torch.float32, device=dev)
    out = torch.full((n,), float("nan"), dtype=torch.float32, device=dev)
    lp = torch.zeros(n // 4 + 2, dtype=torch.float32, device=dev)
    s = torch.cuda.current_stream(dev).cuda_stream
    got = []
    for _ in range(2):
        g = torch.full_like(p, float("nan"))
        ND._abi.check(L.nd_mp_forward(n, rp.data_ptr(), nb.data_ptr(), af.data_ptr(), Xd.data_ptr(), nfeat, p.data_ptr(),
                                      work.data_ptr(), out.data_ptr(), s))
        ND._abi.check(L.nd_mp_backward(n, rp.data_ptr(), nb.data_ptr(), ab.data_ptr(), Xd.data_ptr(), nfeat, p.data_ptr(),
                                       yd.data_ptr(), work.data_ptr(), g.data_ptr(), lp.data_ptr(), s))
        got.append((out.cpu().numpy().copy(), g.cpu().numpy()))
    ref_out, _ = mpnn_ref.forward(params, X, A)
    loss, gref = mpnn_ref.loss_and_grad(params, X, A, y)
    np.testing.assert_allclose(got[0][0], ref_out, rtol=2e-4, atol=2e-5)
    assert np.linalg.norm(got[0][1] - gref) <= 2e-4 * np.linalg.norm(gref)
    assert abs(lp.sum().item() / n - loss) <= 1e-4 * loss
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("copies", [40, 80, 16400])
def test_copies_of_a_graph(ND, dev, copies):
    """A node's output depends on its row's entries alone and is formed in the same order in
    every launch shape: the copies' outputs equal the graph's bit for bit.  The loss is a mean, so
    the gradients are the graph's up to the rounding of longer sums."""
    import torch
    n0, nfeat = 513, 8
    A, params, X, y = _problem(n0, nfeat)
    rows = np.repeat(np.arange(n0), np.diff(A.indptr))
    d = lambda x, dt: torch.from_numpy(np.ascontiguousarray(x, dt)).to(dev)
    p, L = d(params, np.float32), ND._abi.lib()
    s = torch.cuda.current_stream(dev).cuda_stream

    def run(m):
        n, nnz = m * n0, A.nnz
        k = torch.arange(m, dtype=torch.int32, device=dev)[:, None]
        rp = torch.cat([(d(A.indptr[:-1], np.int32)[None] + nnz * k).reshape(-1),
                        torch.tensor([m * nnz], dtype=torch.int32, device=dev)])
        nb = (d(A.indices, np.int32)[None] + n0 * k).reshape(-1)
        af, ab = d(A.data, np.float32).repeat(m), d(A.toarray().T[rows, A.indices], np.float32).repeat(m)
        Xd, yd = d(X, np.float32).repeat(m, 1), d(y, np.float32).repeat(m)
        work = torch.empty(int(L.nd_mp_workspace_floats(n)), dtype=torch.float32, device=dev)
        out, g = torch.empty(n, dtype=torch.float32, device=dev), torch.empty_like(p)
        lp = torch.zeros(n // 4 + 2, dtype=torch.float32, device=dev)
        ND._abi.check(L.nd_mp_forward(n, rp.data_ptr(), nb.data_ptr(), af.data_ptr(), Xd.data_ptr(), nfeat, p.data_ptr(),
                                      work.data_ptr(), out.data_ptr(), s))
        ND._abi.check(L.nd_mp_backward(n, rp.data_ptr(), nb.data_ptr(), ab.data_ptr(), Xd.data_ptr(), nfeat, p.data_ptr(),
                                       yd.data_ptr(), work.data_ptr(), g.data_ptr(), lp.data_ptr(), s))
        return out, g.cpu().numpy()

    out1, g1 = run(1)
    outm, gm = run(copies)
    assert torch.equal(outm.reshape(copies, n0), out1[None].expand(copies, n0))
    assert np.linalg.norm(gm - g1) <= 2e-4 * np.linalg.norm(g1)
