"""Batched personalised PageRank in groups of 32 columns: every column is the
scalar loop's, bit for bit and with its iteration count, on rows around every
edge of the kernels' splits (8-edge steps, tiles, 1024-edge hubs, hub chunks),
vertices without in- or out-edges, every group and hub width, and scores small
enough that contributions are subnormal."""
import numpy as np
import pytest

import oracle
from gardenia_ocl_amd import PersonalizedPageRankPlan

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 255, 256, 257, 767, 768, 769, 1023, 1024, 1025,
           1151, 1152, 1153, 2305, 4096, 4097]


def _csr(m, rows):
    off = np.zeros(m + 1, np.int32)
    off[1:] = np.cumsum([len(r) for r in rows])
    return off, np.concatenate([np.asarray(r, np.int32) for r in rows]).astype(np.int32)


def _lengths_graph(m=6001):
    """Every length of LENGTHS several times between short rows; only the first
    5000 vertices have out-edges."""
    rng = np.random.default_rng(5)
    n = rng.integers(0, 12, m)
    n[rng.permutation(m)[:4 * len(LENGTHS)]] = np.tile(LENGTHS, 4)
    return _csr(m, [np.sort(rng.choice(5000, size=k, replace=False)) for k in n])


def _layers_graph(layers=14, leaves=3000):
    """p0 -> p1 -> ..., every p also to all leaves: after i steps a p's share of
    the seed's mass is (0.85 / 3001)^i, below the smallest normal float from i = 11."""
    m = layers + leaves
    return _csr(m, [[r - 1] if 0 < r < layers else list(range(layers)) if r >= layers else []
                    for r in range(m)])


def _run(device, off, col, seeds, k, tol, max_iter, chunk, **kw):
    import torch

    m = len(off) - 1
    deg = np.bincount(col, minlength=m).astype(np.int32)
    keep = [torch.from_numpy(a).to(device) for a in (off, col, deg)]
    plan = PersonalizedPageRankPlan(*keep, k, **kw)
    X = plan.one_hot(seeds)
    st, _, _ = plan.run(torch.from_numpy(seeds).to(device), X, tol=tol, max_iter=max_iter,
                        chunk=chunk)
    return X.cpu().numpy(), plan.column_iterations(), deg


@pytest.mark.parametrize("k,kc,hub_cols,relabel,chunk", [
    (64, 0, 0, False, 1), (64, 64, 16, True, 3), (192, 64, 64, False, 2), (256, 256, 32, True, 1),
    (128, 128, 0, False, 0)])
def test_ppr_groups_bit_exact(device, k, kc, hub_cols, relabel, chunk):
    off, col = _lengths_graph()
    m = len(off) - 1
    rng = np.random.default_rng(k)
    seeds = rng.integers(0, 5000, k).astype(np.int32)
    stop = rng.random(k) < 0.6
    seeds[stop] = rng.integers(5000, m, int(stop.sum()))  # no out-edges: 2 iterations
    X, its, deg = _run(device, off, col, seeds, k, 1e-5, 60, chunk, k_chunk=kc, hub_cols=hub_cols,
                       relabel=relabel)
    for j in range(k):
        ref, it, _ = oracle.ppr(m, off, col, deg, int(seeds[j]), tol=1e-5, max_iter=60)
        np.testing.assert_array_equal(X[:, j], ref)
        assert its[j] == it


@pytest.mark.parametrize("relabel", [False, True])
def test_ppr_subnormal_contributions(device, relabel):
    off, col = _layers_graph()
    m, k = len(off) - 1, 64
    seeds = (np.arange(k) % 14).astype(np.int32)
    X, _, deg = _run(device, off, col, seeds, k, 0.0, 16, 0, relabel=relabel)
    tiny = np.finfo(np.float32).tiny
    assert ((X > 0) & (X / np.maximum(deg, 1)[:, None] < tiny)).any()
    for j in range(14):
        ref, _, _ = oracle.ppr(m, off, col, deg, int(seeds[j]), tol=0.0, max_iter=16)
        np.testing.assert_array_equal(X[:, j], ref)
    np.testing.assert_array_equal(X[:, 14:28], X[:, :14])


@pytest.mark.parametrize("edges", [0, 1])
def test_ppr_hardly_any_edges(device, edges):
    """No row with edges at all, or a single one."""
    m, k = 37, 64
    off = np.zeros(m + 1, np.int32)
    off[20:] = edges
    col = np.full(edges, 3, np.int32)
    seeds = (np.arange(k) % m).astype(np.int32)
    X, its, deg = _run(device, off, col, seeds, k, 1e-6, 20, 1)
    for j in range(m):
        ref, it, _ = oracle.ppr(m, off, col, deg, j, tol=1e-6, max_iter=20)
        np.testing.assert_array_equal(X[:, j], ref)
        assert its[j] == it
