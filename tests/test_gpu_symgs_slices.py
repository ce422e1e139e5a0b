"""SymGS short rows in slices of up to 64 (uniform and general), bit for bit
with the oracle's sequential sweep: rows of 0 .. 65 off-diagonal entries, every
remainder of the stored groups, colors of 1, 63, 64, 65 and more rows, rows
without a diagonal, and an x that holds infinities that no padding may touch."""
import numpy as np
import pytest

import oracle
from gardenia_ocl_amd import SymGSPlan, graph

pytestmark = pytest.mark.gpu


def _csr(m, rows):
    off = np.zeros(m + 1, np.int32)
    col = []
    for r in range(m):
        col.extend(sorted(rows[r]))
        off[r + 1] = len(col)
    return off, np.array(col, np.int32)


def _banded(m, offsets, diag):
    """Row r holds r + d for every offset d inside the matrix."""
    return _csr(m, [[r + d for d in offsets if 0 <= r + d < m] + ([r] if diag(r) else [])
                    for r in range(m)])


def _mixed(m, rng):
    """Rows of 0 .. 65 entries at random columns; some without a diagonal."""
    rows = []
    for r in range(m):
        c = set(rng.choice(m, size=int(rng.integers(0, 66)), replace=False).tolist())
        (c.add if r % 5 else c.discard)(r)
        rows.append(c)
    return _csr(m, rows)


@pytest.mark.parametrize("kind", ["band1", "band5", "band64", "mixed", "tiny"])
def test_symgs_slices_bit_exact(device, kind):
    import torch

    rng = np.random.default_rng(7)
    if kind == "mixed":
        m = 700
        off, col = _mixed(m, rng)
    elif kind == "tiny":
        m = 1
        off, col = _csr(m, [[0]])
    else:
        half = {"band1": [1], "band5": [1, 3, 4, 9, 70], "band64": list(range(1, 33))}[kind]
        m = {"band1": 130, "band5": 64 * 10 + 1, "band64": 64 * 33 + 63}[kind]
        offs = sorted(half + [-d for d in half] + ([200] if kind == "band5" else []))
        off, col = _banded(m, offs, lambda r: r % 50 != 3)
    val = graph.uniform_pm1(len(col), 11).astype(np.float32)
    for r in range(m):
        val[off[r]:off[r + 1]][col[off[r]:off[r + 1]] == r] = 40.0
    # first-fit coloring over the symmetrized pattern
    adj = [set() for _ in range(m)]
    for r in range(m):
        for j in col[off[r]:off[r + 1]]:
            if j != r:
                adj[r].add(int(j))
                adj[int(j)].add(r)
    color = np.full(m, -1)
    for r in range(m):
        used = {color[j] for j in adj[r]}
        color[r] = next(c for c in range(m + 1) if c not in used)
    idx = np.argsort(color, kind="stable").astype(np.int32)
    co = np.concatenate([[0], np.cumsum(np.bincount(color))]).astype(np.int32)
    b = graph.uniform_pm1(m, 5).astype(np.float32)
    for with_inf in (False, True):
        x0 = graph.uniform_pm1(m, 3).astype(np.float32)
        if with_inf:
            x0[[0, m // 2]] = [np.inf, -np.inf]  # column 0 and an inner one
        with np.errstate(all="ignore"):
            want = oracle.symgs(off, col, idx, val, x0, b, co, 2)
        t = [torch.from_numpy(a).to(device) for a in (off, col, val, idx)]
        plan = SymGSPlan(*t, co)
        x = torch.from_numpy(x0).to(device)
        plan.run(x, torch.from_numpy(b).to(device), 2)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(x.cpu().numpy(), want)
