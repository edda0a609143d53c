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
