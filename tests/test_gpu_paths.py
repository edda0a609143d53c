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


def _with_filler(inputs, B, rows):
    """The batch with one cell more: a diagonal of `rows` rows without nodes, solved at once."""
    ro, rp, col, val, no, en, ec, nrhs, po, pi, pw, pc = inputs
    n, k = int(ro[-1]), np.arange(rows)
    out = (np.append(ro, n + rows), np.concatenate([rp, rp[-1] + 1 + k]).astype(np.int32),
           np.concatenate([col, n + k]).astype(np.int32), np.concatenate([val, np.full(rows, 2.0 + 0.5j)]),
           np.append(no, no[-1]), np.concatenate([en.reshape(-1), np.full(2 * rows, -1)]).astype(np.int32),
           np.concatenate([ec.reshape(-1), np.zeros(2 * rows)]), nrhs, np.concatenate([po, np.full(nrhs, po[-1])]), pi, pw,
           np.concatenate([pc, np.zeros(nrhs)]))
    return out, np.concatenate([B, np.ones((rows, nrhs))])


@pytest.mark.parametrize("nrhs", [1, 2])
def test_cell_result_does_not_depend_on_the_batch(torch_dev, nrhs):
    """Cells of one to three row tiles alone and beside a cell of 250 k and of 1.7 M rows (one, two
    and all sub-tiles of a tile per block): the sums of a cell are the same in every batch, so its
    solution, iterations and residual are, bit for bit."""
    from edgefem_amd import _capi
    from test_gpu_parity import _ragged_cells
    inputs, B, Xref = _ragged_cells([700, 1024, 1500, 2100], nrhs=nrhs, seed=5)
    n, ref = B.shape[0], None
    for rows in (0, 250_000, 1_700_000):
        cells, rhs = _with_filler(inputs, B, rows) if rows else (inputs, B)
        batch = _capi.CellBatch(*cells)
        X, iters, resid = batch.solve(torch_dev.from_numpy(rhs).cuda(), tol=1e-12)
        X = X.cpu().numpy().reshape(-1, nrhs)
        batch.close()
        print(f"nrhs {nrhs}, {rows} rows beside: iterations {iters[:4].ravel()}", flush=True)
        assert resid.max() <= 1e-12
        if rows:
            np.testing.assert_array_equal(X[n:], rhs[n:] / (2.0 + 0.5j))
        got = X[:n], iters[:4], resid[:4]
        ref = ref or got
        for a, b in zip(got, ref):
            np.testing.assert_array_equal(a, b)


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
    for variant, cap in ((-1, 1000), (-1, 7), (0, 7)):
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
        assert s.spmv_variant()[0] == variant   # -1: nothing was timed, the one kernel ran
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
    d = np.abs(X[-1, 7] - X[0, 7]).max() / np.abs(X[0, 7]).max()
    print(f"    7 iterations, one kernel against one launch per step: {d:.1e}", flush=True)
    assert d <= max(1e-13, n * 2.3e-16)


@pytest.mark.parametrize("n,nrhs,dtype,terms", [
    (600, 8, "complex128", 0), (600, 2, "complex64", 0), (600, 2, "complex128", 3), (600, 3, "complex128", 0),
    (140000, 2, "complex128", 0)])
def test_systems_past_the_persistent_kernel(torch_dev, n, nrhs, dtype, terms):
    """What the one kernel does not cover (more right-hand sides, single precision, more
    terms, more rows) is solved by the timed forms.  Bound: the tolerance, 1e-6 for values
    rounded to single precision (2^-24 of rows whose entries sum to less than 4 times the diagonal)."""
    import torch
    from edgefem_amd import _capi
    A, en, B = _local_system(n, nrhs, 1)
    rows, w, c = _lowrank_terms(n, 3, np.random.default_rng(2))
    s = _capi.KrylovSolver(A.indptr, A.indices, nrhs=nrhs, dtype=getattr(torch, dtype))
    if terms:
        s.set_lowrank(rows.reshape(-1), w.reshape(-1), c)
    s.set_matrix(torch.from_numpy(A.data).to(getattr(torch, dtype)))
    X, info = s.solve(torch.from_numpy(B).cuda(), tol=1e-10)
    X = X.cpu().numpy().reshape(n, nrhs)
    r = B - A @ X
    for p in range(terms):
        k = rows[p] >= 0
        r[rows[p][k]] -= c[p] * np.outer(w[p][k], w[p][k].conj() @ X[rows[p][k]])
    assert info["converged"] and s.spmv_variant()[0] >= 0
    assert np.linalg.norm(r) <= (2e-10 if dtype == "complex128" else 1e-6) * np.linalg.norm(B)


@pytest.mark.parametrize("kind,rows,entries,one_kernel", [
    ("one long row", 1500, 256, True), ("one long row", 1500, 257, False), ("one long row", 1500, 1100, False),
    ("all rows", 900, 96, True), ("all rows", 900, 97, False)])
def test_persistent_kernel_by_row_length(torch_dev, kind, rows, entries, one_kernel):
    """The longest row and the mean row at their limits and one entry past them; longer rows go to
    the timed variants, as before there was one kernel.  Tolerance as in test_persistent_cocg_edges."""
    import scipy.sparse as sp
    import torch
    from edgefem_amd import _capi
    rng = np.random.default_rng(entries)
    k = np.arange(rows)
    if kind == "all rows":   # a ring of `entries` columns centred on the row (one more past it where even)
        off = [d for d in range(1, (entries - 1) // 2 + 1)]
        A = sum(sp.csr_matrix((np.full(rows, 0.1 + 0.02j), (k, (k + d) % rows)), shape=(rows, rows)) for d in off)
        A = A + A.T
        if entries % 2 == 0:
            A = A + sp.csr_matrix((np.full(rows, 0.1), (k, (k + rows // 2) % rows)), shape=(rows, rows))
    else:
        r = rows // 2
        j = np.delete(np.arange(r - entries // 2, r - entries // 2 + entries), entries // 2)
        A = sp.csr_matrix((np.full(entries - 1, 0.05 + 0.01j), (np.full(entries - 1, r), j)), shape=(rows, rows))
        A = A + A.T
    A = (A + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel() * 1.6 + 1.0)).tocsr()
    A.sort_indices()
    assert np.diff(A.indptr).max() == entries and (kind != "all rows" or A.nnz == rows * entries)
    B = rng.standard_normal((rows, 2)) + 1j * rng.standard_normal((rows, 2))
    s = _capi.KrylovSolver(A.indptr, A.indices, nrhs=2)
    s.set_matrix(A.data)
    X, info = s.solve(torch.from_numpy(B).cuda(), tol=1e-12)
    rel = np.linalg.norm(B - A @ X.cpu().numpy().reshape(B.shape)) / np.linalg.norm(B)
    assert info["converged"] and rel <= 2e-12 and (s.spmv_variant()[0] == -1) == one_kernel


def _persistent_case(n, nrhs, aux, terms):
    """Solver, right-hand sides (one of zeros) and what a residual needs."""
    import torch
    from edgefem_amd import _capi
    A, en, B = _local_system(n, nrhs, n + 7, long_rows=(0, n - 1))
    if nrhs > 1:
        B[:, 0] = 0
    lr = _lowrank_terms(n, terms, np.random.default_rng(n)) if terms else None

    def solver():
        s = _capi.KrylovSolver(A.indptr, A.indices, nrhs=nrhs)
        if aux:
            s.set_gradient(_Nodes(en))
        if lr:
            s.set_lowrank(lr[0].reshape(-1), lr[1].reshape(-1), lr[2])
        s.set_matrix(A.data)
        return s

    def residual(X):
        X = X.cpu().numpy().reshape(n, nrhs)
        r = B - A @ X
        for p in range(terms):
            k = lr[0][p] >= 0
            r[lr[0][p][k]] -= lr[2][p] * np.outer(lr[1][p][k], lr[1][p][k].conj() @ X[lr[0][p][k]])
        return np.linalg.norm(r) / np.linalg.norm(B)

    return solver, torch.from_numpy(B).cuda(), residual


@pytest.mark.parametrize("n,nrhs,aux,terms", [
    (700, 2, True, 0), (700, 2, True, 2), (700, 1, False, 3), (1100, 4, True, 0), (70000, 2, True, 1),
    (70000, 1, False, 0)])
@pytest.mark.parametrize("per_launch", [1, 5, 8])
def test_persistent_kernel_over_several_launches(torch_dev, n, nrhs, aux, terms, per_launch):
    """Iterations split over launches (odd and even numbers of them: p alternates between two
    copies) are the ones of a single launch: bit for bit, with low-rank terms to the rounding
    of w^H p, formed again at each launch (30 iterations of sums of 9 terms, below 1e-13 of x
    times the condition number, below 10)."""
    import torch
    solver, b, residual = _persistent_case(n, nrhs, aux, terms)
    for cap in (12, 1000):
        one, many = solver(), solver()
        many.set_persist_limits(per_launch)
        X, i1 = one.solve(b, tol=1e-12, max_iterations=cap)
        Y, i2 = many.solve(b, tol=1e-12, max_iterations=cap)
        assert one.spmv_variant()[0] == many.spmv_variant()[0] == -1
        if terms and cap == 1000:
            assert i2["converged"] and residual(Y) <= 2e-12 and abs(max(i1["iters"]) - max(i2["iters"])) <= 1
        else:
            np.testing.assert_array_equal(i1["iters"], i2["iters"])
        d = (X - Y).abs().max().item() / X.abs().max().item()
        print(f"n {n} nrhs {nrhs} terms {terms} cap {cap}: iterations {i1['iters']} {i2['iters']} difference {d:.1e}",
              flush=True)
        assert d <= 1e-12 if terms else torch.equal(X, Y)


@pytest.mark.parametrize("n,nrhs,aux,terms", [(700, 2, True, 0), (700, 1, False, 3), (70000, 2, True, 1)])
def test_persistent_kernel_that_gives_up(torch_dev, n, nrhs, aux, terms):
    """With no poll at all every block leaves its first wait at once: the solve starts again with
    launches per step on the buffers that the kernel has written, and later solves of this
    solver do not try it again, until the limits are set."""
    import torch
    solver, b, residual = _persistent_case(n, nrhs, aux, terms)
    s, fresh = solver(), solver()
    s.set_persist_limits(polls=0)
    X, info = s.solve(b, tol=1e-12)
    v = s.spmv_variant()[0]
    assert v >= 0 and info["converged"] and residual(X) <= 2e-12
    if nrhs > 1:
        assert X.reshape(n, nrhs)[:, 0].abs().max().item() == 0
    fresh.set_spmv_variant(v)
    Y, _ = fresh.solve(b, tol=1e-12)
    assert torch.equal(X, Y)
    X, info = s.solve(b, tol=1e-12)
    assert s.spmv_variant()[0] == v and torch.equal(X, Y)
    s.set_persist_limits()
    X, info = s.solve(b, tol=1e-12)
    assert s.spmv_variant()[0] == -1 and info["converged"] and residual(X) <= 2e-12


def test_persistent_kernels_of_several_threads(torch_dev):
    """Solvers whose blocks take all CUs, half of them and a few, in four threads on streams of
    their own: no launch keeps another from its CUs (a wait that gave up would leave launches
    per step), and every result is the one of a solver alone, bit for bit."""
    import threading
    import torch
    sizes = [(65536, 1), (65400, 2), (30000, 2), (700, 2)]
    cases = [_persistent_case(n, nrhs, False, 0) for n, nrhs in sizes]
    ref = [solver().solve(b, tol=1e-12)[0] for solver, b, _ in cases]
    solvers = [c[0]() for c in cases]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(30):
                X, _ = solvers[i].solve(cases[i][1], tol=1e-12)
                if not torch.equal(X, ref[i]) or solvers[i].spmv_variant()[0] != -1:
                    bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_tuned_solver_keeps_the_persistent_kernel(torch_dev):
    """A profiled solve and one with too many low-rank terms time the variants; what they chose does
    not change a later solve that the one kernel covers: the same bits as a fresh solver's."""
    import torch
    from edgefem_amd import _capi
    n = 600
    A, en, B = _local_system(n, 2, 4)
    rows, w, c = _lowrank_terms(n, 3, np.random.default_rng(2))
    b = torch.from_numpy(B).cuda()

    def solver():
        s = _capi.KrylovSolver(A.indptr, A.indices, nrhs=2)
        s.set_gradient(_Nodes(en))
        s.set_matrix(A.data)
        return s

    ref, _ = solver().solve(b, tol=1e-12)
    s = solver()
    s.profile(True)
    s.solve(b, tol=1e-12)
    assert s.spmv_variant()[0] >= 0
    s.profile(False)
    X, info = s.solve(b, tol=1e-12)
    assert s.spmv_variant()[0] == -1 and info["converged"] and torch.equal(X, ref)
    s = solver()
    s.set_lowrank(rows.reshape(-1), w.reshape(-1), c)   # 3 terms and 2 right-hand sides: not covered
    s.set_matrix(A.data)
    s.solve(b, tol=1e-12)
    assert s.spmv_variant()[0] >= 0
    s.set_lowrank(rows[:0].reshape(-1), w[:0].reshape(-1), c[:0])
    s.set_matrix(A.data)
    X, info = s.solve(b, tol=1e-12)
    assert s.spmv_variant()[0] == -1 and info["converged"] and torch.equal(X, ref)
    s.set_spmv_variant(0)
    assert s.spmv_variant()[0] == 0
    s.solve(b, tol=1e-12)
    assert s.spmv_variant()[0] == 0


def _fan_mesh(levels, ring):
    """Tetrahedra around an axis: axis edges with 3 ring + 1 entries in their rows, axis nodes
    of degree 2 ring + 2."""
    ang = 2 * np.pi * np.arange(ring) / ring
    xyz = [(0.0, 0.0, float(k)) for k in range(levels + 1)]
    tets = []
    for k in range(levels):
        base = len(xyz)
        xyz += [(np.cos(t), np.sin(t), k + 0.5) for t in ang]
        tets += [(k, k + 1, base + i, base + (i + 1) % ring) for i in range(ring)]
    return np.array(xyz), np.array(tets)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("nsys,levels,ring,lossy,packed", [
    (1, 3, 7, False, False), (2, 40, 9, True, False), (18, 5, 60, False, False), (39, 4, 30, True, False),
    (65, 2, 30, False, False), (95, 3, 20, False, False), (143, 2, 60, True, False),
    (32, 33, 30, False, False), (65, 32, 30, False, False), (65, 33, 30, False, True), (95, 33, 30, True, True),
    (96, 33, 30, False, False), (143, 33, 30, True, True), (144, 33, 30, False, False),
    (1, 34, 60, False, True), (2, 270, 9, True, True), (18, 34, 60, False, True), (32, 67, 30, True, True),
    (33, 67, 30, True, False), (95, 34, 60, True, True), (129, 34, 60, False, True), (136, 67, 30, True, True),
    (38, 134, 30, False, True), (39, 134, 30, False, False), (88, 134, 30, True, True), (89, 134, 30, False, False),
    (143, 67, 60, True, True), (144, 67, 60, False, False)])
def test_packed_sweep_batches(torch_dev, nsys, levels, ring, lossy, packed, graph):
    """Sweeps whose systems are packed into wavefronts, and those on the other side of the rule
    (fewer rows, more systems): one system to three wavefronts of them, chunks with more
    entries than are staged, real and complex matrices, two ports, a right-hand side of zeros,
    eager and replayed.  tol = 1e-10; the recursive residual drifts from the true one by
    iterations (below 400 on the meshes of more than 6,000 rows) times eps times the condition of
    the scaled matrix (below 1e3), 0.9e-10: 2e-10 in all.  After 5 iterations the result agrees
    with the padded kernels to the rounding of 5 sums of n terms times that condition, below
    1e-9."""
    import torch
    import scipy.sparse as sp
    from edgefem_amd import _capi
    xyz, tets = _fan_mesh(levels, ring)
    topo = _capi.Topology(np.arange(len(xyz)), tets, np.zeros((0, 3), np.int32))
    n = topo.n_edges
    rng = np.random.default_rng(nsys)
    eps = np.full(len(tets), 2.0 - 0.3j if lossy else 2.0 + 0j)
    K, M = _capi.assemble_km(topo, xyz, eps)
    ptr, col = topo.row_ptr.cpu().numpy(), topo.col_idx.cpu().numpy()
    row = np.repeat(np.arange(n), np.diff(ptr))
    Ms = [np.where((row == col) & (row % 9 == 2 * p), 0.5, 0.0) for p in range(2)]
    k2 = -rng.uniform(1.0, 3.0, nsys)
    coef = rng.uniform(0.1, 1.0, (nsys, 2)) * (1 + 0.2j)
    B = rng.standard_normal((n, nsys)) + 1j * rng.standard_normal((n, nsys))
    if nsys > 1:
        B[:, nsys // 2] = 0
    X = {}
    for pinned in (False, True):
        sweep = _capi.SweepSolver(topo, K, M, [torch.from_numpy(m).cuda() for m in Ms], None, nsys)
        if pinned:
            sweep.set_variants(1, 1)
        sweep.set_graph(graph)
        for cap in (10000, 5):
            X[pinned, cap], info = sweep.solve(k2, coef, torch.from_numpy(B).cuda(), tol=1e-10, max_iterations=cap)
            X[pinned, cap] = X[pinned, cap].cpu().numpy().reshape(n, nsys)
            if cap == 10000:
                iters = info["iters"]
        got = sweep.variants()[:2]
        assert got == (1, 1) if pinned else (got == (-1, -1)) == packed
    csr = lambda v: sp.csr_matrix((v, col, ptr), shape=(n, n))   # noqa: E731
    Y = X[False, 10000]
    r = B - csr(K.cpu().numpy()) @ Y + (csr(M.cpu().numpy()) @ Y) * k2
    for p in range(2):
        r -= (csr(Ms[p]) @ Y) * coef[:, p]
    on = np.linalg.norm(B, axis=0) > 0
    rel = (np.linalg.norm(r, axis=0)[on] / np.linalg.norm(B, axis=0)[on]).max()
    d = np.abs(X[False, 5] - X[True, 5]).max() / np.abs(X[True, 5]).max()
    print(f"n {n} nsys {nsys}: iterations {iters.max()} true {rel:.1e}; 5 iterations against padded {d:.1e}", flush=True)
    assert iters.max() < 400 and rel <= 2e-10 and np.all(Y[:, ~on] == 0)
    assert d <= 1e-9


@pytest.mark.parametrize("graph", [False, True])
def test_narrow_batch_after_a_wide_one(torch_dev, graph):
    """A narrow batch on a sweep that has solved a wide one is packed as on a new sweep, with the
    same bits, and a wide one after it runs what was chosen; pinned variants stay pinned."""
    import torch
    from edgefem_amd import _capi
    xyz, tets = _fan_mesh(34, 60)
    topo = _capi.Topology(np.arange(len(xyz)), tets, np.zeros((0, 3), np.int32))
    n = topo.n_edges
    rng = np.random.default_rng(3)
    K, M = _capi.assemble_km(topo, xyz, np.full(len(tets), 2.0 - 0.3j))
    k2 = -rng.uniform(1.0, 3.0, 128)
    B = torch.from_numpy(rng.standard_normal((n, 128)) + 1j * rng.standard_normal((n, 128))).cuda()

    def sweep():
        s = _capi.SweepSolver(topo, K, M, [], None, 128)
        s.set_graph(graph)
        return s

    def solve(s, m):
        X, info = s.solve(k2[:m], np.zeros((m, 0)), B[:, :m].contiguous(), tol=1e-10, max_iterations=1000)
        assert info["resid"].max() <= 1e-10
        return X

    ref = solve(sweep(), 18)
    s = sweep()
    solve(s, 128)
    wide = s.variants()[:2]
    assert min(wide) >= 0
    X = solve(s, 18)
    assert s.variants()[:2] == (-1, -1) and torch.equal(X, ref)
    solve(s, 128)
    assert s.variants()[:2] == wide
    s.set_variants(1, 1)
    solve(s, 18)
    assert s.variants()[:2] == (1, 1)


@pytest.mark.parametrize("n,nrhs,kind", [
    (5, 1, "real"), (511, 2, "mixed"), (512, 1, "complex"), (513, 2, "real"), (1600, 2, "mixed"), (9000, 1, "mixed"),
    (40000, 2, "scattered"), (3000, 2, "long")])
def test_staged_spmv_tiles(torch_dev, n, nrhs, kind):
    """SpMV variant 11 with tiles of 512 rows: a last tile of one row, wavefronts without rows,
    real and complex tiles side by side, rows of 250 entries, columns that do not fit (then
    without staging); a second matrix on the same solver.  True residual as in
    test_persistent_cocg_edges; 7 iterations against one launch per row group likewise."""
    import scipy.sparse as sp
    import torch
    from edgefem_amd import _capi
    A, en, B = _local_system(n, nrhs, n + 1, long_rows=(0, n // 2, n - 1))
    rng = np.random.default_rng(n)
    if kind == "scattered":
        perm = rng.permutation(n)
        A = A[perm][:, perm].tocsr()
    elif kind == "long":
        j = np.arange(n // 2 + 1, n // 2 + 225)
        far = sp.csr_matrix((np.full(j.size, 0.01 + 0.01j), (np.full(j.size, n // 2), j)), shape=(n, n))
        A = (A + far + far.T + 6 * sp.identity(n)).tocsr()
    A.sort_indices()
    mats = [A]
    if kind in ("real", "mixed"):
        half = n if kind == "real" else n // 2
        Ar = A.copy()
        row = np.repeat(np.arange(n), np.diff(A.indptr))
        Ar.data = np.where((row < half) & (A.indices < half), np.abs(A.data.real) * np.sign(A.data.real), A.data)
        Ar = (Ar + sp.diags(np.asarray(abs(A).sum(axis=1)).ravel())).tocsr()
        Ar.sort_indices()
        mats = [Ar, A] if kind == "mixed" else [Ar]
    s = _capi.KrylovSolver(A.indptr, A.indices, nrhs=nrhs)
    s.set_gradient(_Nodes(en))
    b = torch.from_numpy(B).cuda()
    for Am in mats:
        assert np.array_equal(Am.indices, A.indices)
        s.set_matrix(Am.data)
        X = {}
        for variant, cap in ((11, 1000), (11, 7), (0, 7)):
            s.set_spmv_variant(variant)
            X[variant, cap], info = s.solve(b, tol=1e-12, max_iterations=cap)
            X[variant, cap] = X[variant, cap].cpu().numpy().reshape(n, nrhs)
            if cap == 1000:
                rel = (np.linalg.norm(B - Am @ X[variant, cap], axis=0) / np.linalg.norm(B, axis=0)).max()
                print(f"n {n} {kind}: iterations {max(info['iters'])} true {rel:.1e}", flush=True)
                assert info["converged"] and rel <= 2e-12
                assert s.staged() == (kind != "scattered")
        d = np.abs(X[11, 7] - X[0, 7]).max() / np.abs(X[0, 7]).max()
        assert d <= max(1e-13, n * 2.3e-16), d
        assert not s.staged()   # variant 0 ran last


def _spread_system(n, reach, nrhs, seed):
    """A diagonally dominant matrix whose rows couple up to `reach` away, eight entries to a side."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(n), 8)
    j = i + rng.integers(1, reach, i.size)
    ok = j < n
    off = sp.csr_matrix((rng.standard_normal(ok.sum()) + 0.1j, (i[ok], j[ok])), shape=(n, n))
    off = off + off.T
    A = (off + sp.diags(np.asarray(abs(off).sum(axis=1)).ravel() * 1.6 + 1.0)).tocsr()
    A.sort_indices()
    return A, rng.standard_normal((n, nrhs)) + 1j * rng.standard_normal((n, nrhs))


def test_staged_solvers_of_different_tiles(torch_dev):
    """The LDS limit of a kernel belongs to all solvers: one of large tiles (more than 64 KiB of
    columns) solves before and after another of small ones is built, with the same bits."""
    import torch
    from edgefem_amd import _capi

    def make(reach):
        A, B = _spread_system(4000, reach, 2, reach)
        s = _capi.KrylovSolver(A.indptr, A.indices, nrhs=2)
        s.set_matrix(A.data)
        s.set_spmv_variant(11)
        tiles = [A[r:r + 512] for r in range(0, 4000, 512)]
        return s, torch.from_numpy(B).cuda(), max(np.unique(t.indices).size for t in tiles) * 32

    large, b, lds = make(1000)
    assert 65536 < lds < 80 * 1024
    X, info = large.solve(b, tol=1e-12)
    assert info["converged"] and large.staged()
    small, b2, lds = make(40)
    assert lds < 32768
    Y, info = small.solve(b2, tol=1e-12)
    assert info["converged"] and small.staged()
    X2, info = large.solve(b, tol=1e-12)
    assert info["converged"] and large.staged() and torch.equal(X, X2)


@pytest.mark.parametrize("nrhs", [1, 2])
def test_staged_tile_at_the_most_columns(torch_dev, nrhs):
    """The first tile reads exactly the columns that leave room for two blocks in the 160 KiB of a
    CU (80 KiB less 16 bytes per wavefront and right-hand side of two), and one more: staged and
    not, both solved."""
    import scipy.sparse as sp
    import torch
    from edgefem_amd import _capi
    most = (80 * 1024 - 8 * 2 * 16) // (16 * nrhs)
    rng = np.random.default_rng(nrhs)
    for cols in (most, most + 1):
        extra, n = cols - 512, cols + 100
        off = sp.csr_matrix((np.full(extra, 0.2 + 0.1j), (np.arange(extra) % 512, 512 + np.arange(extra))), shape=(n, n))
        A = (off + off.T + sp.diags(np.full(n, 4.0 + 1j))).tocsr()
        A.sort_indices()
        B = rng.standard_normal((n, nrhs)) + 1j * rng.standard_normal((n, nrhs))
        s = _capi.KrylovSolver(A.indptr, A.indices, nrhs=nrhs)
        s.set_matrix(A.data)
        s.set_spmv_variant(11)
        X, info = s.solve(torch.from_numpy(B).cuda(), tol=1e-12)
        rel = np.linalg.norm(B - A @ X.cpu().numpy().reshape(B.shape)) / np.linalg.norm(B)
        assert info["converged"] and rel <= 2e-12 and s.staged() == (cols == most)


def test_staged_spmv_needs_few_right_hand_sides(torch_dev):
    """With three right-hand sides variant 11 runs on split values, and the persistent kernel is
    not reported as staged."""
    import torch
    from edgefem_amd import _capi
    for nrhs, variant, staged in ((3, 11, False), (2, 11, True), (2, -1, False)):
        A, en, B = _local_system(900, nrhs, 5)
        s = _capi.KrylovSolver(A.indptr, A.indices, nrhs=nrhs)
        s.set_gradient(_Nodes(en))
        s.set_matrix(A.data)
        s.set_spmv_variant(variant)
        X, info = s.solve(torch.from_numpy(B).cuda(), tol=1e-12)
        rel = np.linalg.norm(B - A @ X.cpu().numpy().reshape(B.shape)) / np.linalg.norm(B)
        assert info["converged"] and rel <= 2e-12 and s.staged() == staged


@pytest.mark.parametrize("grid", [1, 3, 4, 6, 9, 10])
def test_edge_numbering_of_large_buckets(torch_dev, grid):
    """Cones of 2 grid^2 tetrahedra over a square: the apex, lowest id, has 6 grid^2 edge slots
    (6 to 600: one, two, four entries per lane of the sort, and past it).  Edges in first-seen
    order and signs, whole numbers, against a scan in Python."""
    from edgefem_amd import _capi
    node = lambda i, j: 1 + i * (grid + 1) + j   # noqa: E731
    tets = []
    for i in range(grid):
        for j in range(grid):
            a, b, c, d = node(i, j), node(i + 1, j), node(i, j + 1), node(i + 1, j + 1)
            tets += [(a, b, d, 0), (c, a, 0, d)]
    rng = np.random.default_rng(grid)
    tets = np.array(tets)[rng.permutation(len(tets))]
    ids = np.concatenate([[5], 7 + rng.permutation((grid + 1) ** 2)]).astype(np.int64)
    seen, edges, sign = {}, np.zeros((len(tets), 6), int), np.zeros((len(tets), 6), int)
    for t, tet in enumerate(tets):
        for l, (p, q) in enumerate(((0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3))):
            a, b = ids[tet[p]], ids[tet[q]]
            edges[t, l] = seen.setdefault((min(a, b), max(a, b)), len(seen))
            sign[t, l] = 1 if a < b else -1
    topo = _capi.Topology(ids, tets, np.zeros((0, 3), np.int32))
    assert topo.n_edges == len(seen)
    np.testing.assert_array_equal(topo.edges.cpu().numpy(), np.array(list(seen)))
    np.testing.assert_array_equal(topo.tet_edges.cpu().numpy(), edges)
    np.testing.assert_array_equal(topo.tet_sign.cpu().numpy(), sign)


def test_assembly_scratch_from_two_threads(torch_dev):
    """Assemblies of one mesh from two threads on two streams share its scratch only one at a
    time: every result is the single-threaded one, bit for bit."""
    import threading
    import torch
    from edgefem_amd import _capi
    xyz, tets = _fan_mesh(400, 50)
    topo = _capi.Topology(np.arange(len(xyz)), tets, np.zeros((0, 3), np.int32))
    scales = [1.0, 1.5]
    ref = [[v.clone() for v in _capi.assemble_km(topo, xyz * c, np.full(len(tets), 2.0 + 0j))] for c in scales]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                K, M = _capi.assemble_km(topo, xyz * scales[i], np.full(len(tets), 2.0 + 0j))
                if not (torch.equal(K, ref[i][0]) and torch.equal(M, ref[i][1])):
                    bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("levels,keeps", [(20000, True), (65000, False)])
def test_assembly_scratch_is_bounded(torch_dev, levels, keeps):
    """An assembly's scratch (336 bytes per tet) stays with the mesh up to 1 GiB and is freed beyond:
    what the device has less after an assembly, apart from torch's own pool, is the scratch (320 MiB)
    or nothing (of 1,041), give or take tens of MiB that the runtime takes and returns by itself:
    on which side of half the scratch it lies."""
    import torch
    from edgefem_amd import _capi
    ring = 50
    ang = 2 * np.pi * np.arange(ring) / ring
    k, i = (v.ravel() for v in np.meshgrid(np.arange(levels), np.arange(ring), indexing="ij"))
    xyz = np.concatenate([np.stack([np.zeros(levels + 1), np.zeros(levels + 1), np.arange(levels + 1.0)], 1),
                          np.stack([np.cos(ang)[i], np.sin(ang)[i], k + 0.5], 1)])
    base = levels + 1 + k * ring
    tets = np.stack([k, k + 1, base + i, base + (i + 1) % ring], 1).astype(np.int32)
    topo = _capi.Topology(np.arange(len(xyz)), tets, np.zeros((0, 3), np.int32))
    scratch = len(tets) * 336
    assert (scratch <= 2 ** 30) == keeps
    xyz0, tets0 = _fan_mesh(3, 7)
    small = _capi.Topology(np.arange(len(xyz0)), tets0, np.zeros((0, 3), np.int32))
    _capi.assemble_km(small, xyz0, np.full(len(tets0), 2.0 + 0j))   # the runtime's first allocations
    torch.cuda.synchronize()
    held = lambda: -torch.cuda.mem_get_info()[0] - torch.cuda.memory_reserved()   # noqa: E731
    before = held()
    for _ in range(2):
        K, M = _capi.assemble_km(topo, xyz, np.full(len(tets), 2.0 + 0j))
    torch.cuda.synchronize()
    got = held() - before
    print(f"{len(tets)} tets: scratch {scratch / 2**20:.0f} MiB, held after {got / 2**20:.0f} MiB", flush=True)
    assert (got > scratch / 2) == keeps
