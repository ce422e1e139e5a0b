"""Plans that gather through windows of their source vector and plans that do
not: which one a graph or matrix gets by its size and by how far its sources
are spread, and that every option gives the plain sequential result.

Windows are checked bit for bit: PageRank and SpMV against the oracle; weighted
PageRank against its sequential sums, the adjoint on values whose sums are
exact in FP32 in any order."""
import numpy as np
import pytest

import oracle
from gardenia_ocl_amd import PageRankPlan, SpmvPlan
from gardenia_ocl_amd.autograd import SpmvBackwardPlan, WeightedPageRankPlan

pytestmark = pytest.mark.gpu

LINE = 1 << 21


def _t(device, a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).to(device)


def _in_csr(m, src, dst):
    order = np.argsort(dst, kind="stable")
    off = np.zeros(m + 1, np.int32)
    np.cumsum(np.bincount(dst, minlength=m), out=off[1:])
    return off, src[order].astype(np.int32)


def _graph(m, form, rng):
    n = m // 2
    src, dst = rng.integers(0, m, n), rng.integers(0, m, n)
    if form == "gaps":  # sources in the second, the last and every fourth window
        w = src // 32768
        src = np.where((w % 4 == 0) | (w == 1) | (w == (m - 1) // 32768), src, (src + 32768 * 4 - w % 4 * 32768) % m)
    elif form == "hubs":  # hub rows of one staging block, exactly one, and several
        dst[:17194] = np.concatenate([np.full(4096, 7), np.full(4097, m - 1), np.full(9001, m // 2)])
    off, col = _in_csr(m, src, dst)
    return off, col, np.maximum(np.bincount(col, minlength=m), 1).astype(np.int32)


def _near(m, k, rng):
    """k sources per row within 500 of it, in order."""
    col = (np.arange(m)[:, None] + np.sort(rng.integers(-500, 500, (m, k)), 1)) % m
    return (np.arange(m + 1) * k).astype(np.int32), col.astype(np.int32).ravel()


@pytest.mark.parametrize("m", [LINE + 1, LINE + 32767])
@pytest.mark.parametrize("form", ["spread", "gaps", "hubs"])
def test_pagerank_options_through_windows(device, m, form):
    rng = np.random.default_rng(m)
    off, col, deg = _graph(m, form, rng)
    args = _t(device, off), _t(device, col), _t(device, deg)
    init = rng.random(m).astype(np.float32) / np.float32(m)
    ref, _, _ = oracle.pr(m, off, col, deg, init, tol=0.0, max_iter=3)
    one = np.zeros(m, np.float32)
    seed = int(col[0])
    one[seed] = 1.0
    seeded = None
    for kw in ({"stage_hubs": 0}, {}, {"stage_hubs": 1}, {"block": 512}, {"block": 1024},
               {"items_per_thread": 8}, {"hub_threshold": 64}, {"nontemporal": 2}):
        plan = PageRankPlan(*args, relabel=False, **kw)
        assert plan.windowed == ("stage_hubs" not in kw or kw["stage_hubs"] != 0)
        for _ in range(2):  # direct launches, then the captured graph
            s = _t(device, init)
            plan.run(s, tol=0.0, max_iter=3)
            np.testing.assert_array_equal(s.cpu().numpy(), ref, err_msg=str(kw))
        s = _t(device, one)
        plan.run(s, tol=0.0, max_iter=3, seed_vertex=seed)
        seeded = s.cpu().numpy() if seeded is None else seeded  # the plain gather's
        np.testing.assert_array_equal(s.cpu().numpy(), seeded, err_msg=str(kw))
        plan.close()


def test_relabelled_pagerank_through_windows(device):
    m = (7 << 20) + 1
    rng = np.random.default_rng(m)
    off, col, deg = _graph(m, "hubs", rng)
    init = rng.random(m).astype(np.float32) / np.float32(m)
    ref, _, _ = oracle.pr(m, off, col, deg, init, tol=0.0, max_iter=3)
    for kw, on in (({"relabel": True}, True), ({}, True), ({"relabel": True, "stage_hubs": 0}, False)):
        plan = PageRankPlan(_t(device, off), _t(device, col), _t(device, deg), **kw)
        assert plan.windowed == on
        s = _t(device, init)
        plan.run(s, tol=0.0, max_iter=3)
        np.testing.assert_array_equal(s.cpu().numpy(), ref, err_msg=str(kw))
        plan.close()


@pytest.mark.parametrize("m", [LINE + 1, LINE + 32769])
def test_weighted_pagerank_through_windows(device, m):
    """Out-weights of every vertex sum to 4 (4096 for five vertices of many
    out-edges), so divisions by them are exact; the cotangent is 0 or 1, and
    two adjoint iterations with damping 1/2 need at most 24 bits."""
    import torch

    rng = np.random.default_rng(m)
    hubs = np.array([0, 5, 40000, m // 2, m - 1])
    plain = np.setdiff1d(np.arange(m), hubs)
    src = np.concatenate([np.repeat(plain, 4), np.repeat(hubs, 4096)])
    a = np.tile(np.array([0.5, 1.0, 1.0, 1.5], np.float32), len(src) // 4)
    dst = plain[rng.integers(0, len(plain), len(src))]
    dst[:9001] = plain[77]       # in-edge hubs: three staging blocks, and one
    dst[20000:24096] = plain[-3]
    order = np.argsort(dst, kind="stable")
    off, col = _in_csr(m, src, dst)
    a = a[order]
    s = np.where(np.isin(np.arange(m), hubs), np.float32(4096), np.float32(4))
    plan = WeightedPageRankPlan(_t(device, off), _t(device, col), _t(device, a))
    assert plan.windowed == (True, True)
    # forward: sequential sums of rounded products
    x = rng.random(m).astype(np.float32) / np.float32(m)
    dx = _t(device, x)
    damp = np.float32(0.5)
    base = (np.float32(1.0) - damp) / np.float32(m)
    for _ in range(3):
        x = base + damp * oracle.spmv(m, off, col, a, x / s, np.zeros(m, np.float32))
    st = plan.forward(dx, damping=0.5, tol=0.0, max_iter=3)
    assert st["iterations"] == 3
    np.testing.assert_array_equal(dx.cpu().numpy(), x)
    # adjoint: exact
    w = rng.integers(0, 2, m).astype(np.float32)
    row = np.repeat(np.arange(m), np.diff(off))
    lam = w.astype(np.float64)
    for _ in range(2):
        lam = w + 0.5 * np.bincount(col, weights=a * lam[row], minlength=m) / s
    q = (np.bincount(col, weights=a * lam[row], minlength=m) / s).astype(np.float32)
    lam = lam.astype(np.float32)
    dlam = torch.empty_like(dx)
    grad = torch.empty(len(col), dtype=torch.float32, device=device)
    plan.backward(dx, _t(device, w), dlam, grad, damping=0.5, tol=0.0, max_iter=2)
    np.testing.assert_array_equal(dlam.cpu().numpy(), lam)
    np.testing.assert_array_equal(grad.cpu().numpy(), damp * (x / s)[col] * (lam[row] - q[col]))


def test_sources_near_their_rows_stay_out_of_windows(device):
    import torch

    rng = np.random.default_rng(11)
    for m, k, relabel in ((LINE + 5, 3, False), ((7 << 20) + 5, 3, None)):
        off, col = _near(m, k, rng)
        deg = np.maximum(np.bincount(col, minlength=m), 1).astype(np.int32)
        plan = PageRankPlan(_t(device, off), _t(device, col), _t(device, deg), relabel=relabel)
        assert not plan.windowed
        init = rng.random(m).astype(np.float32) / np.float32(m)
        s = _t(device, init)
        plan.run(s, tol=0.0, max_iter=2)
        ref, _, _ = oracle.pr(m, off, col, deg, init, tol=0.0, max_iter=2)
        np.testing.assert_array_equal(s.cpu().numpy(), ref)
        plan.close()
    m, k = LINE + 5, 8
    off, col = _near(m, k, rng)
    val = rng.random(m * k, dtype=np.float32) - np.float32(0.5)
    assert WeightedPageRankPlan(_t(device, off), _t(device, col),
                                _t(device, np.abs(val))).windowed == (False, False)
    x = rng.random(m, dtype=np.float32)
    plan = SpmvPlan(_t(device, off), _t(device, col), _t(device, val), m)
    assert not plan.windowed
    y = torch.zeros(m, device=device)
    plan.run(_t(device, x), y)
    np.testing.assert_array_equal(y.cpu().numpy(),
                                  oracle.spmv(m, off, col, val, x, np.zeros(m, np.float32)))
    bwd = SpmvBackwardPlan(_t(device, off), _t(device, col), m)
    assert not bwd.windowed
    g = rng.random(m, dtype=np.float32) - np.float32(0.5)
    row = np.repeat(np.arange(m), k)
    dx, dA = torch.empty(m, device=device), torch.empty(m * k, device=device)
    bwd.run(_t(device, val), _t(device, x), _t(device, g), dx, dA)
    np.testing.assert_array_equal(dA.cpu().numpy(), g[row] * x[col])
    order = np.argsort(col, kind="stable")
    toff = np.zeros(m + 1, np.int32)
    np.cumsum(np.bincount(col, minlength=m), out=toff[1:])
    np.testing.assert_array_equal(
        dx.cpu().numpy(), oracle.spmv(m, toff, row[order].astype(np.int32), val[order], g,
                                      np.zeros(m, np.float32)))


@pytest.mark.parametrize("rows,cols,k,on", [
    ((LINE >> 2) + 9, LINE + 9, 2, True),    # half a nonzero per column
    ((LINE >> 2) - 9, LINE + 9, 2, False),
    (1 << 20, LINE - 9, 2, False),           # one, where two are asked for
    (1 << 20, (1 << 20) + 9, 3, True),
    (1 << 20, 1 << 20, 3, False),            # x fits the L2
])
def test_spmv_lines(device, rows, cols, k, on):
    import torch

    rng = np.random.default_rng(rows)
    off = (np.arange(rows + 1) * k).astype(np.int32)
    col = rng.integers(0, cols, rows * k).astype(np.int32)
    val = rng.random(rows * k, dtype=np.float32) - np.float32(0.5)
    x = rng.random(cols, dtype=np.float32)
    g = rng.random(rows, dtype=np.float32)
    plan = SpmvPlan(_t(device, off), _t(device, col), _t(device, val), cols, mode="auto")
    bwd = SpmvBackwardPlan(_t(device, off), _t(device, col), cols)
    assert plan.windowed == on and bwd.windowed == on
    y = torch.zeros(rows, device=device)
    plan.run(_t(device, x), y)
    np.testing.assert_array_equal(y.cpu().numpy(),
                                  oracle.spmv(rows, off, col, val, x, np.zeros(rows, np.float32)))
    dA = torch.empty(rows * k, device=device)
    bwd.run(_t(device, val), _t(device, x), _t(device, g), None, dA)
    np.testing.assert_array_equal(dA.cpu().numpy(), np.repeat(g, k) * x[col])
