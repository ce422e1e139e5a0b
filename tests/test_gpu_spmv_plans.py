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


@pytest.mark.parametrize("rows,cols,lens", [
    (60000, (1 << 20) + 77, [40]),                     # x through windows
    (3000, 5000, [2049, 1500, 0, 9000, 700]),          # long rows beside the tiles
    (3000, (1 << 20) + 77, [2049, 1500, 0, 9000, 700]),  # both
])
def test_two_threads_run_one_plan(device, rows, cols, lens):
    """Every run gives its own x's result, whichever threads queue runs meanwhile."""
    import threading

    import torch

    rng = np.random.default_rng(rows)
    lens = np.resize(np.asarray(lens), rows)
    Ap = np.zeros(rows + 1, np.int32)
    np.cumsum(lens, out=Ap[1:])
    nnz = int(Ap[-1])
    Aj = rng.integers(0, cols, nnz).astype(np.int32)
    Ax = rng.random(nnz, dtype=np.float32) - np.float32(0.5)
    row = np.repeat(np.arange(rows), lens)
    dAp, dAj, dAx = _t(device, Ap), _t(device, Aj), _t(device, Ax)
    plan = SpmvPlan(dAp, dAj, dAx, cols)
    bwd = SpmvBackwardPlan(dAp, dAj, cols)
    runs, threads = 40, 2
    x = [rng.random(cols, dtype=np.float32) - np.float32(0.5) for _ in range(threads)]
    g = [rng.random(rows, dtype=np.float32) - np.float32(0.5) for _ in range(threads)]
    dx_in, dg = [_t(device, a) for a in x], [_t(device, a) for a in g]
    ys = [torch.zeros(runs, rows, dtype=torch.float32, device=device) for _ in range(threads)]
    dA = [torch.empty(4, nnz, dtype=torch.float32, device=device) for _ in range(threads)]
    dx = [torch.empty(4, cols, dtype=torch.float32, device=device) for _ in range(threads)]
    torch.cuda.synchronize()
    start = threading.Barrier(threads)

    def work(i):
        start.wait()
        for r in range(runs):
            plan.run(dx_in[i], ys[i][r])
        for r in range(4):
            bwd.run(dAx, dx_in[i], dg[i], dx[i][r], dA[i][r])

    ts = [threading.Thread(target=work, args=(i,)) for i in range(threads)]
    for th in ts:
        th.start()
    for th in ts:
        th.join()
    torch.cuda.synchronize()
    order = np.argsort(Aj, kind="stable")
    toff = np.zeros(cols + 1, np.int32)
    np.cumsum(np.bincount(Aj, minlength=cols), out=toff[1:])
    for i in range(threads):
        ref = _t(device, oracle.spmv(rows, Ap, Aj, Ax, x[i], np.zeros(rows, np.float32)))
        assert bool((ys[i] == ref).all())
        assert bool((dA[i] == _t(device, g[i][row] * x[i][Aj])).all())
        ref = _t(device, oracle.spmv(cols, toff, row[order].astype(np.int32), Ax[order], g[i],
                                     np.zeros(cols, np.float32)))
        assert bool((dx[i] == ref).all())
