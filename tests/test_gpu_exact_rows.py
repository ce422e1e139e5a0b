"""Row sums of PageRank-like plans against the sequential FP32 loop, bit for
bit, at the row lengths where the way of adding changes (the owner thread's
chain, a wavefront's 256- and 1024-term passes, a workgroup's 4096-term
chunks) and with terms that are hard for it: ties, terms of every exponent,
subnormals, long runs of zeros, a few or many negative terms, inf."""
import numpy as np
import pytest

import oracle
from gardenia_ocl_amd import MultiGraphPageRank, PageRankPlan

pytestmark = pytest.mark.gpu

LENS = [31, 33, 64, 511, 512, 513, 575, 576, 577, 767, 769, 1023, 1025, 1088, 1600, 2047, 2500,
        4095, 4096, 4097, 5119, 8192, 8193, 12291]
KINDS = ["uniform", "ties", "wide", "tiny", "zeros", "few_negative", "signs", "inf", "halves"]


def _terms(kind, n, rng):
    v = rng.random(n).astype(np.float32)
    if kind == "ties":  # whole and half ulps of a sum that starts at 2^23 of them
        v = rng.choice(np.array([0.5, 1.0, 1.5, 2.5, 0.25], np.float32), n)
        v[0] = 2.0 ** 23
    elif kind == "halves":
        v = np.full(n, 0.5, np.float32)
        v[0] = 2.0 ** 23 + 1
    elif kind == "wide":
        v = np.exp2(rng.uniform(-60, 30, n)).astype(np.float32)
    elif kind == "tiny":
        v = (rng.integers(0, 50, n) * np.float32(1e-45)).astype(np.float32)
        v[n // 2:] = np.float32(1.2e-38) * rng.random(n - n // 2).astype(np.float32)
    elif kind == "zeros":
        v[: n - 7] = 0.0
        v[n // 3] = 1.0
    elif kind == "few_negative":
        v[:: max(1, n // 3)] *= -1
    elif kind == "signs":
        v -= np.float32(0.5)
    elif kind == "inf":
        v[n - n // 4] = np.inf
    return v


def _graph(kind):
    """Rows of LENS, each over leaves of its own whose contribution is the term."""
    rng = np.random.default_rng(KINDS.index(kind))
    k, total = len(LENS), sum(LENS)
    m = k + total
    off = np.full(m + 1, total, np.int32)
    off[0] = 0
    off[1:k + 1] = np.cumsum(LENS)
    leaves = rng.permutation(total)
    col = (k + leaves).astype(np.int32)
    init = np.zeros(m, np.float32)
    at = 0
    for n in LENS:
        init[col[at:at + n]] = _terms(kind, n, rng)
        at += n
    return m, off, col, np.ones(m, np.int32), init


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("kw", [{}, {"relabel": True}, {"hub_threshold": 64}, {"sort_tiles": False},
                                {"items_per_thread": 8, "relabel": True}, {"block": 512}])
def test_rows_are_the_sequential_sums(device, kind, kw):
    import torch

    m, off, col, deg, init = _graph(kind)
    ref, _, _ = oracle.pr(m, off, col, deg, init, tol=0.0, max_iter=1)
    t = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
    plan = PageRankPlan(t(off), t(col), t(deg), **kw)
    s = t(init.copy())
    plan.run(s, tol=0.0, max_iter=1)
    plan.close()
    np.testing.assert_array_equal(s.cpu().numpy(), ref)


@pytest.mark.parametrize("kind", ["uniform", "ties", "wide", "signs"])
def test_rows_of_many_graphs(device, kind):
    import torch

    m, off, col, deg, init = _graph(kind)
    ref, _, _ = oracle.pr(m, off, col, deg, init, tol=0.0, max_iter=1)
    t = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
    g = (t(off), t(col), t(deg))
    small = (t(np.array([0, 1, 2], np.int32)), t(np.array([1, 0], np.int32)),
             t(np.ones(2, np.int32)))
    plan = MultiGraphPageRank([g, small, g])
    s = [t(init.copy()), t(np.full(2, 0.5, np.float32)), t(init.copy())]
    plan.run(s, tol=0.0, max_iter=1)
    plan.close()
    np.testing.assert_array_equal(s[0].cpu().numpy(), ref)
    np.testing.assert_array_equal(s[2].cpu().numpy(), ref)
