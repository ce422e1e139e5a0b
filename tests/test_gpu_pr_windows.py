"""Plans whose gathers go through windows of sources (more than 2^20
vertices), against the oracle and the plain gather, bit for bit: vertex counts
around a window's 32,768 sources, empty windows, hub rows of one and several
staging blocks, personalised runs, both tile widths."""
import numpy as np
import pytest

import oracle
from gardenia_ocl_amd import PageRankPlan

pytestmark = pytest.mark.gpu

BASE = 1 << 20


def _graph(m, form, rng):
    n = m // 2
    if form == "spread":
        src, dst = rng.integers(0, m, n), rng.integers(0, m, n)
    elif form == "ends":  # only the first and the last window are gathered from
        src = np.where(rng.random(n) < 0.5, rng.integers(0, 100, n), m - 1 - rng.integers(0, 100, n))
        dst = rng.integers(0, m, n)
    else:  # hubs of one staging block, exactly one, and several
        src = rng.integers(0, m, n)
        dst = np.concatenate([np.full(4096, 7), np.full(4097, m - 1), np.full(9001, m // 2),
                              rng.integers(0, m, n - 17194)])
    order = np.argsort(dst, kind="stable")
    src, dst = src[order].astype(np.int32), dst[order]
    off = np.zeros(m + 1, np.int32)
    np.cumsum(np.bincount(dst, minlength=m), out=off[1:])
    deg = np.maximum(np.bincount(src, minlength=m), 1).astype(np.int32)
    return off, src, deg


@pytest.mark.parametrize("m", [BASE + 1, BASE + 32767, BASE + 32768, BASE + 32769, BASE + 100003])
@pytest.mark.parametrize("form", ["spread", "ends", "hubs"])
def test_windows_match_oracle_and_plain_gather(device, m, form):
    import torch

    rng = np.random.default_rng(m)
    off, col, deg = _graph(m, form, rng)
    t = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
    args = t(off), t(col), t(deg)
    init = rng.random(m).astype(np.float32) / np.float32(m)
    ref, _, _ = oracle.pr(m, off, col, deg, init, tol=0.0, max_iter=3)
    for kw in ({}, {"relabel": True}, {"block": 512}, {"items_per_thread": 8}, {"stage_hubs": 0},
               {"hub_threshold": 64}):
        plan = PageRankPlan(*args, **kw)
        for _ in range(2):  # direct launches, then the captured graph
            s = t(init.copy())
            plan.run(s, tol=0.0, max_iter=3)
            np.testing.assert_array_equal(s.cpu().numpy(), ref, err_msg=str(kw))
        plan.close()
    seed = int(col[0])
    one = np.zeros(m, np.float32)
    one[seed] = 1.0
    got = []
    for kw in ({}, {"stage_hubs": 0}):
        plan = PageRankPlan(*args, **kw)
        s = t(one.copy())
        plan.run(s, tol=0.0, max_iter=3, seed_vertex=seed)
        got.append(s.cpu().numpy())
        plan.close()
    np.testing.assert_array_equal(got[0], got[1])


@pytest.mark.parametrize("m,relabel", [((1 << 21) + 1, False), ((1 << 21) + 32769, False),
                                       ((7 << 20) + 1, True), ((7 << 20) + 32768, True)])
@pytest.mark.parametrize("form", ["spread", "ends", "hubs"])
def test_windows_past_their_lines(device, m, relabel, form):
    import torch

    rng = np.random.default_rng(m)
    off, col, deg = _graph(m, form, rng)
    t = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
    init = rng.random(m).astype(np.float32) / np.float32(m)
    ref, _, _ = oracle.pr(m, off, col, deg, init, tol=0.0, max_iter=3)
    for kw in ({}, {"block": 512}, {"hub_threshold": 64}):
        plan = PageRankPlan(t(off), t(col), t(deg), relabel=relabel, **kw)
        for _ in range(2):  # direct launches, then the captured graph
            s = t(init.copy())
            plan.run(s, tol=0.0, max_iter=3)
            np.testing.assert_array_equal(s.cpu().numpy(), ref, err_msg=str(kw))
        plan.close()
