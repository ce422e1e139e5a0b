"""SpMV and its backward where x goes through windows (more than 2^20
columns), against the oracle's sequential loop, bit for bit: column counts
around a window's 32,768, rows around a tile's 2048 nonzeros, long rows beside
the tiles and inside their launch, unsorted and repeated columns, empty rows
and matrices whose columns use few windows."""
import numpy as np
import pytest

import oracle
from gardenia_ocl_amd import SpmvPlan
from gardenia_ocl_amd.autograd import SpmvBackwardPlan

pytestmark = pytest.mark.gpu

BASE = 1 << 20


def _matrix(rows, cols, lens, form, rng):
    lens = np.resize(np.asarray(lens), rows)
    off = np.zeros(rows + 1, np.int32)
    np.cumsum(lens, out=off[1:])
    nnz = int(off[-1])
    if form == "ends":
        col = np.where(rng.random(nnz) < 0.5, rng.integers(0, 9, nnz),
                       cols - 1 - rng.integers(0, 9, nnz))
    else:
        col = rng.integers(0, cols, nnz)
    if form == "sorted":
        row = np.repeat(np.arange(rows), lens)
        col = col[np.lexsort((col, row))]
    return off, col.astype(np.int32), (rng.random(nnz, dtype=np.float32) - np.float32(0.5))


CASES = [
    # rows, cols, row lengths (repeated over the rows), form
    (1200, BASE + 1, [2047, 2048, 0, 1999, 3000], "random"),          # long rows, one launch
    (3000, BASE + 32767, [2049, 1500, 0, 9000, 700], "random"),       # long rows, side stream
    (70001, BASE + 32768, [31, 0, 64, 33, 1, 65, 17], "sorted"),
    (70001, BASE + 32769, [31, 0, 64, 33, 1, 65, 17], "ends"),
    (2100000, BASE + 100003, [1, 0, 2, 3, 0, 0, 1], "random"),        # tiles full of rows
    (3000, 5000, [2049, 1500, 0, 9000, 700], "random"),               # side stream, no windows
    (1200, BASE + 1, [3000], "random"),                               # long rows only
]


@pytest.mark.parametrize("rows,cols,lens,form", CASES)
def test_windowed_spmv_and_backward(device, rows, cols, lens, form):
    import torch

    rng = np.random.default_rng(rows)
    Ap, Aj, Ax = _matrix(rows, cols, lens, form, rng)
    x = rng.random(cols, dtype=np.float32) - np.float32(0.5)
    y0 = rng.random(rows, dtype=np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
    dAp, dAj, dAx, dx_in = t(Ap), t(Aj), t(Ax), t(x)
    ref = oracle.spmv(rows, Ap, Aj, Ax, x, y0.copy())
    for mode in ("tiles", "auto"):
        plan = SpmvPlan(dAp, dAj, dAx, cols, mode=mode)
        for _ in range(2):
            y = t(y0)
            plan.run(dx_in, y)
            np.testing.assert_array_equal(y.cpu().numpy(), ref)
        dAx.mul_(-2.0)  # the values are read on every call
        plan.refresh_values()
        y = t(np.zeros(rows, np.float32))
        plan.run(dx_in, y)
        np.testing.assert_array_equal(
            y.cpu().numpy(), oracle.spmv(rows, Ap, Aj, Ax * np.float32(-2), x,
                                         np.zeros(rows, np.float32)))
        dAx.mul_(-0.5)
        plan.close()
    g = rng.random(rows, dtype=np.float32) - np.float32(0.5)
    row = np.repeat(np.arange(rows), np.diff(Ap))
    bwd = SpmvBackwardPlan(dAp, dAj, cols)
    dx = torch.empty(cols, dtype=torch.float32, device=device)
    dA = torch.empty(len(Aj), dtype=torch.float32, device=device)
    bwd.run(dAx, dx_in, t(g), dx, dA)
    np.testing.assert_array_equal(dA.cpu().numpy(), g[row] * x[Aj])
    order = np.argsort(Aj, kind="stable")
    toff = np.zeros(cols + 1, np.int32)
    np.cumsum(np.bincount(Aj, minlength=cols), out=toff[1:])
    np.testing.assert_array_equal(
        dx.cpu().numpy(), oracle.spmv(cols, toff, row[order].astype(np.int32), Ax[order], g,
                                      np.zeros(cols, np.float32)))
    bwd.close()
