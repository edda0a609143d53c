"""GPU tests of kernel paths chosen by size, each at the sizes where it can go wrong."""

import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available()
    torch.cuda.set_device(0)
    return torch


@pytest.mark.parametrize("nrhs", [1, 2])
@pytest.mark.parametrize("sizes", [[64], [30, 65, 128, 129], [700, 26, 257]])
def test_cell_batch_tile_edges_vs_dense_solve(torch_dev, sizes, nrhs):
    """Cells whose rows end at, before and after a tile of the batch kernels (64 rows, 1,024
    entries, 64 nodes), against a dense LU of every cell.  The cells are diagonally
    dominant (condition number below 10), so a residual of 1e-12 bounds the relative error
    by 1e-11."""
    from edgefem_amd import _capi
    from test_gpu_parity import _ragged_cells
    inputs, B, Xref = _ragged_cells(sizes, nrhs=nrhs, seed=11)
    batch = _capi.CellBatch(*inputs)
    Bd = torch_dev.from_numpy(B).cuda()
    X, iters, resid = batch.solve(Bd, tol=1e-12)
    err = np.abs(X.cpu().numpy().reshape(B.shape) - Xref).max() / np.abs(Xref).max()
    print(f"sizes {sizes} nrhs {nrhs}: iterations {iters.ravel()} err {err:.1e}", flush=True)
    assert resid.max() <= 1e-12 and iters.max() < 100
    assert err <= 1e-11
    batch.close()


def _local_system(n, nrhs, seed, long_rows=()):
    """A complex-symmetric, diagonally dominant matrix (condition number below 10) whose
    rows couple to neighbours at most 40 away, 5 to 15 entries each and about 40 in
    long_rows, with end nodes of every row for the nodal preconditioner (-1 rows included)."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(n), 4)
    j = i + rng.integers(1, 41, i.size)
    for r in long_rows:
        i = np.concatenate([i, np.full(36, r)])
        j = np.concatenate([j, r + np.arange(-18, 18) * 2 + 1])
    ok = (j >= 0) & (j < n) & (i != j)
    v = rng.standard_normal(ok.sum()) + 1j * rng.standard_normal(ok.sum())
    off = sp.csr_matrix((v, (i[ok], j[ok])), shape=(n, n))
    off = off + off.T
    dom = np.asarray(abs(off).sum(axis=1)).ravel() * 1.6 + 1.0
    A = (off + sp.diags(dom * np.exp(0.4j))).tocsr()
    A.sort_indices()
    en = np.stack([np.arange(n) // 5, np.arange(n) // 5 + 1 + np.arange(n) % 3], axis=1).astype(np.int32)
    B = rng.standard_normal((n, nrhs)) + 1j * rng.standard_normal((n, nrhs))
    return A, en, B


class _Nodes:
    def __init__(self, en):
        self.n_nodes = int(en.max()) + 1
        flat = en.reshape(-1)
        order = np.argsort(flat, kind="stable")
        ptr = np.concatenate([[0], np.cumsum(np.bincount(flat, minlength=self.n_nodes))])
        from edgefem_amd._capi import to_dev
        import torch
        self.edge_nodes = to_dev(en.reshape(-1), torch.int32)
        self.n2e_ptr = to_dev(ptr.astype(np.int32), torch.int32)
        self.n2e = to_dev((order // 2).astype(np.int32), torch.int32)


def _lowrank_terms(n, count, rng):
    """count disjoint real vectors of 9 rows each (the last padded), and their coefficients."""
    rows = rng.choice(n, size=(count, 9), replace=False).astype(np.int32)
    w = rng.standard_normal((count, 9)).astype(np.complex128)
    rows[-1, 5:] = -1
    return rows, w, 0.7 + 0.2j * np.arange(1, count + 1)


@pytest.mark.parametrize("n,nrhs,aux,terms", [
    (33, 1, True, 0), (255, 1, False, 4), (256, 2, True, 0), (257, 2, True, 2), (1025, 3, True, 0),
    (1025, 4, True, 0), (3000, 1, True, 3), (65536, 2, False, 0), (65537, 2, True, 1), (65664, 1, True, 0),
    (131072, 2, True, 0)])
def test_persistent_cocg_edges(torch_dev, n, nrhs, aux, terms):
    """COCG in one kernel at the edges of its rows per block (256, and more in LDS past
    65,536 rows on 256 CUs), with rows longer than a lane group's registers, each number of
    right-hand sides, with and without the nodal part and low-rank terms.  A recursive
    residual of 1e-12 leaves a true one of at most 1e-12 plus rounding of the 30-odd updates
    of values of order one (below 1e-13): 2e-12.  Stopped after 7 iterations it agrees with
    one launch per step to the rounding of 7 sums of n terms, n eps < 3e-11."""
    import torch
    from edgefem_amd import _capi
    rng = np.random.default_rng(n)
    A, en, B = _local_system(n, nrhs, n, long_rows=(0, n // 2, n - 1))
    B[:, nrhs - 1] = B[:, nrhs - 1] if nrhs < 3 else 0   # a right-hand side of zeros stays zero
    lr = _lowrank_terms(n, terms, rng) if terms else None
    X = {}
    for variant, cap in ((12, 1000), (12, 7), (0, 7)):
        s = _capi.KrylovSolver(A.indptr, A.indices, nrhs=nrhs)
        if aux:
            s.set_gradient(_Nodes(en), (np.arange(n) % 11 == 3).astype(np.uint8))
        if lr:
            s.set_lowrank(lr[0].reshape(-1), lr[1].reshape(-1), lr[2])
        s.set_matrix(A.data)
        s.set_spmv_variant(variant)
        for _ in range(2):   # the second solve finds the first one's workspace
            X[variant, cap], info = s.solve(torch.from_numpy(B).cuda(), tol=1e-12, max_iterations=cap)
        X[variant, cap] = X[variant, cap].cpu().numpy().reshape(n, nrhs)
        if cap == 1000:
            r = B - A @ X[variant, cap]
            for p in range(terms):
                k = lr[0][p] >= 0
                rows, w = lr[0][p][k], lr[1][p][k]
                r[rows] -= lr[2][p] * np.outer(w, w.conj() @ X[variant, cap][rows])
            on = np.linalg.norm(B, axis=0) > 0
            rel = (np.linalg.norm(r, axis=0)[on] / np.linalg.norm(B, axis=0)[on]).max()
            print(f"n {n} nrhs {nrhs} aux {aux} terms {terms}: iterations {list(info['iters'])} true {rel:.1e}",
                  flush=True)
            assert info["converged"] and rel <= 2e-12
            assert np.all(X[variant, cap][:, ~on] == 0)
        else:
            assert max(info["iters"]) == 7
    d = np.abs(X[12, 7] - X[0, 7]).max() / np.abs(X[0, 7]).max()
    print(f"    7 iterations, one kernel against one launch per step: {d:.1e}", flush=True)
    assert d <= max(1e-13, n * 2.3e-16)


def test_persistent_cocg_refuses_what_it_does_not_cover(torch_dev):
    """Forced on a system outside its range the solve is refused; by default the same system
    is solved by the other forms."""
    import torch
    from edgefem_amd import _capi
    A, en, B = _local_system(600, 8, 1)
    rows, w, c = _lowrank_terms(600, 3, np.random.default_rng(2))
    for nrhs, dtype, terms, method in ((8, torch.complex128, 0, 0), (2, torch.complex64, 0, 0),
                                       (2, torch.complex128, 3, 0), (3, torch.complex128, 0, 0),
                                       (2, torch.complex128, 0, 1)):
        s = _capi.KrylovSolver(A.indptr, A.indices, nrhs=nrhs, dtype=dtype)
        if terms:
            s.set_lowrank(rows.reshape(-1), w.reshape(-1), c)
        s.set_matrix(torch.from_numpy(A.data).to(dtype))
        b = torch.from_numpy(np.ascontiguousarray(B[:, :nrhs])).cuda()
        m = _capi.EFM_METHOD_BICGSTAB if method else _capi.EFM_METHOD_COCG
        s.set_spmv_variant(12)
        with pytest.raises(_capi.EdgeFemError, match="does not fit"):
            s.solve(b, method=m)
        s.set_spmv_variant(-1)
        X, info = s.solve(b, tol=1e-10, method=m)
        assert info["converged"]
