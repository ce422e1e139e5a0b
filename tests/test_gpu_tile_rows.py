"""Rows of one tile around the lengths where a tile's way of adding changes:
the granule loop and the blocks of an owner thread's chain (48 terms), and
tiles whose longest row does or does not turn rows of more than 512 edges over
to wavefronts (1536), full and nearly empty tiles, at every alignment.  Sums
are the oracle's sequential FP32 loop, bit for bit."""
import numpy as np
import pytest

import oracle
from gardenia_ocl_amd import MultiGraphPageRank, PageRankPlan, SpmvPlan

pytestmark = pytest.mark.gpu

ROWS = {
    "short": [0, 1, 2, 3, 4, 5, 7, 0, 8, 9, 15, 16, 17, 31, 33] * 7,
    "around_48": list(range(44, 56)) * 3 + [1, 79, 80, 81, 82, 83, 84, 111, 113] * 4,
    "longest_1535": [3, 512, 513, 600, 1, 1535, 2],
    "longest_1536": [513, 1, 1536, 511, 700],
    "longest_1537": [1, 512, 1537, 513, 2, 600],
    "two_tiles": [1536, 1000, 1500, 60, 1537, 513, 514, 515, 5, 1, 1900],
    "one_row_tile": [4096, 4095, 1, 2],
    "many_rows": [1] * 1500 + [0] * 1500 + [3] * 900,
}


def _terms(kind, n, rng):
    if kind == "ties":
        v = rng.choice(np.array([0.5, 1.0, 1.5, 2.5, 0.25], np.float32), n)
        v[rng.integers(0, n)] = 2.0 ** 23
    elif kind == "signs":
        v = rng.random(n).astype(np.float32) - np.float32(0.5)
    else:
        v = np.exp2(rng.uniform(-20, 10, n)).astype(np.float32)
    return v


def _t(device, a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


def _graph(name, kind):
    """Rows over leaves of their own whose contribution is the term."""
    rng = np.random.default_rng(len(name))
    lens = np.array(ROWS[name])
    k, total = len(lens), int(lens.sum())
    off = np.full(k + total + 1, total, np.int32)
    off[0] = 0
    off[1:k + 1] = np.cumsum(lens)
    leaves = rng.permutation(total).astype(np.int32)
    init = np.zeros(k + total, np.float32)
    init[k + leaves] = _terms(kind, total, rng)
    return k, off, leaves, init


@pytest.mark.parametrize("name", list(ROWS))
@pytest.mark.parametrize("kind", ["ties", "signs", "wide"])
def test_rows_of_a_tile(device, name, kind):
    import torch

    k, off, leaves, init = _graph(name, kind)
    col, m = leaves + k, len(init)
    deg = np.ones(m, np.int32)
    ref, _, _ = oracle.pr(m, off, col, deg, init, tol=0.0, max_iter=1)
    args = _t(device, off), _t(device, col), _t(device, deg)
    for kw in ({}, {"sort_tiles": False}, {"items_per_thread": 8}, {"persistent": True},
               {"block": 512}, {"block": 1024, "relabel": True}):
        plan = PageRankPlan(*args, **kw)
        s = _t(device, init)
        plan.run(s, tol=0.0, max_iter=1)
        np.testing.assert_array_equal(s.cpu().numpy(), ref, err_msg=str(kw))
        plan.close()
    plan = MultiGraphPageRank([args, args])
    s = [_t(device, init), _t(device, init)]
    plan.run(s, tol=0.0, max_iter=1)
    plan.close()
    for a in s:
        np.testing.assert_array_equal(a.cpu().numpy(), ref)
    # SpMV over the same rows, products of the same terms
    Ap, x = off[:k + 1], init[k:]
    Ax = np.where(np.arange(len(leaves)) % 3 == 0, np.float32(-1.25), np.float32(0.75))
    y = np.linspace(-1, 1, k).astype(np.float32)
    plan = SpmvPlan(_t(device, Ap), _t(device, leaves), _t(device, Ax), len(x))
    dy = _t(device, y)
    plan.run(_t(device, x), dy)
    plan.close()
    np.testing.assert_array_equal(dy.cpu().numpy(), oracle.spmv(k, Ap, leaves, Ax, x, y.copy()))
    assert torch.isfinite(dy).all()
