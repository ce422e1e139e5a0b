"""SymGS colors whose rows are sorted by length in chunks of 256 and those
sorted as a whole (14 of 15 rows of one length), bit for bit with
the oracle's sequential sweep: colors around the chunk's and a slice's size,
long rows between the short ones, row lengths around the step widths."""
import numpy as np
import pytest

import oracle
from gardenia_ocl_amd import SymGSPlan, graph

pytestmark = pytest.mark.gpu

C = 3  # color of row r: r % C


def _lens(kind, n, rng):
    if kind == "spread":
        return rng.integers(0, 65, n)
    if kind == "steps":
        return rng.choice([1, 4, 5, 8, 9, 11, 12, 13, 16, 17, 31, 33, 64], n)
    if kind == "long":  # rows of more than 64 entries among the short ones
        return np.where(rng.random(n) < 0.1, rng.integers(65, 200, n), rng.integers(0, 65, n))
    share = {"most": 14 / 15, "below": 0.93, "one_length": 1.0}[kind]
    lens = np.full(n, 14)
    other = rng.permutation(n)[: n - int(np.ceil(share * n))]
    lens[other] = rng.integers(0, 14, len(other))
    return lens


@pytest.mark.parametrize("rows", [63, 255, 256, 257, 513, 1000])
@pytest.mark.parametrize("kind", ["spread", "steps", "long", "most", "below", "one_length"])
def test_symgs_chunks_bit_exact(device, rows, kind):
    import torch

    rng = np.random.default_rng(rows)
    m = C * rows
    lens = np.empty(m, np.int64)
    for c in range(C):
        lens[c::C] = np.minimum(_lens(kind, rows, rng), rows)
    off, col, val = [0], [], []
    for r in range(m):
        # distinct columns of the other colors, near the row where there is room
        near = np.arange(max(0, r - 300), min(m, r + 300))
        near = near[near % C != r % C]
        c = rng.choice(near, size=min(int(lens[r]), len(near)), replace=False)
        c = np.sort(np.append(c, r))
        col.append(c)
        val.append(np.where(c == r, 0.0 if r % 50 == 3 else 90.0, rng.random(len(c)) - 0.5))
        off.append(off[-1] + len(c))
    off = np.array(off, np.int32)
    col = np.concatenate(col).astype(np.int32)
    val = np.concatenate(val).astype(np.float32)
    idx = np.concatenate([np.arange(c, m, C) for c in range(C)]).astype(np.int32)
    co = (np.arange(C + 1) * rows).astype(np.int32)
    x0 = graph.uniform_pm1(m, 3).astype(np.float32)
    b = graph.uniform_pm1(m, 5).astype(np.float32)
    want = oracle.symgs(off, col, idx, val, x0, b, co, 2)
    plan = SymGSPlan(*[torch.from_numpy(a).to(device) for a in (off, col, val, idx)], co)
    x = torch.from_numpy(x0).to(device)
    plan.run(x, torch.from_numpy(b).to(device), 2)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(x.cpu().numpy(), want)
