"""SpMV plans of matrices whose nonzeros all lie in rows longer than a tile
(2048), with empty rows between them, over more than 2^20 columns: the row
tiles hold no nonzero.  Forward in both modes and the backward, whose
transpose has that shape for a tall matrix with an unused column; against the
oracle's sequential loop, bit for bit."""
import numpy as np
import pytest

import oracle
from gardenia_ocl_amd import SpmvPlan
from gardenia_ocl_amd.autograd import SpmvBackwardPlan

pytestmark = pytest.mark.gpu


def _t(device, a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


@pytest.mark.parametrize("rows,lens", [
    (2000, [3000, 0]),              # every second row empty
    (1201, [3000] * 1200 + [0]),    # one empty row at the end
])
@pytest.mark.parametrize("mode", ["tiles", "auto"])
def test_long_rows_and_empty_rows(device, rows, lens, mode):
    rng = np.random.default_rng(rows)
    cols = (1 << 20) + 1
    lens = np.resize(np.asarray(lens), rows)
    Ap = np.zeros(rows + 1, np.int32)
    np.cumsum(lens, out=Ap[1:])
    nnz = int(Ap[-1])
    Aj = rng.integers(0, cols, nnz).astype(np.int32)
    Ax = rng.random(nnz, dtype=np.float32) - np.float32(0.5)
    x = rng.random(cols, dtype=np.float32) - np.float32(0.5)
    y0 = rng.random(rows, dtype=np.float32)
    plan = SpmvPlan(_t(device, Ap), _t(device, Aj), _t(device, Ax), cols, mode=mode)
    y = _t(device, y0)
    plan.run(_t(device, x), y)
    np.testing.assert_array_equal(y.cpu().numpy(), oracle.spmv(rows, Ap, Aj, Ax, x, y0.copy()))


def test_backward_of_a_tall_matrix_with_an_unused_column(device):
    import torch

    rng = np.random.default_rng(5)
    rows, cols, k = (1 << 20) + 3, 1000, 16
    Ap = (np.arange(rows + 1) * k).astype(np.int32)
    Aj = rng.integers(0, cols - 1, rows * k).astype(np.int32)  # never the last column
    Ax = rng.random(rows * k, dtype=np.float32) - np.float32(0.5)
    x = rng.random(cols, dtype=np.float32) - np.float32(0.5)
    g = rng.random(rows, dtype=np.float32) - np.float32(0.5)
    bwd = SpmvBackwardPlan(_t(device, Ap), _t(device, Aj), cols)
    dx = torch.empty(cols, dtype=torch.float32, device=device)
    dA = torch.empty(rows * k, dtype=torch.float32, device=device)
    bwd.run(_t(device, Ax), _t(device, x), _t(device, g), dx, dA)
    row = np.repeat(np.arange(rows), k)
    np.testing.assert_array_equal(dA.cpu().numpy(), g[row] * x[Aj])
    order = np.argsort(Aj, kind="stable")
    toff = np.zeros(cols + 1, np.int32)
    np.cumsum(np.bincount(Aj, minlength=cols), out=toff[1:])
    np.testing.assert_array_equal(
        dx.cpu().numpy(), oracle.spmv(cols, toff, row[order].astype(np.int32), Ax[order], g,
                                      np.zeros(cols, np.float32)))
