"""Plans whose windows do not fit the card's free memory gather plainly, with
the same results; and the failed allocation is not reported by a later call."""
import numpy as np
import pytest

from gardenia_ocl_amd import PageRankPlan, SpmvPlan
from gardenia_ocl_amd.autograd import SpmvBackwardPlan

pytestmark = pytest.mark.gpu

FREE = 600 << 20  # bytes left to the plans


def _fill(torch):
    """Tensors that hold the card's memory but for about FREE bytes."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    held, size = [], 16 << 30
    while size >= 32 << 20:
        if torch.cuda.mem_get_info()[0] - FREE < size:
            size //= 2
            continue
        try:
            held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            size //= 2
    return held


def test_plans_without_room_for_windows(device):
    import torch

    g = torch.Generator(device=device)
    g.manual_seed(1)
    m, k = (1 << 22) + 3, 16  # 67 M entries: 800 MB of windows for SpMV, 400 more for PageRank
    off = torch.arange(m + 1, device=device, dtype=torch.int32) * k
    col = torch.randint(0, m, (m * k,), generator=g, device=device, dtype=torch.int32)
    col[: 5000 * k] = torch.randint(0, m, (5000 * k,), generator=g, device=device)
    # one hub row: its edges taken from the rows behind it
    off[8:6008] = int(off[6008])
    deg = torch.bincount(col, minlength=m).clamp_(min=1).int()
    val = torch.rand(m * k, generator=g, device=device) - 0.5
    x, gr = (torch.rand(m, generator=g, device=device) for _ in range(2))
    y, dA, s = torch.zeros(m, device=device), torch.empty(m * k, device=device), torch.empty(m, device=device)

    def spmv():
        plan = SpmvPlan(off, col, val, m)
        y.zero_()
        plan.run(x, y)
        return plan.windowed, y

    def backward():
        plan = SpmvBackwardPlan(off, col, m)
        plan.run(val, x, gr, None, dA)
        torch.cuda.synchronize()
        return plan.windowed, dA

    def pagerank():
        plan = PageRankPlan(off, col, deg, relabel=False)
        s.fill_(1.0 / m)
        plan.run(s, tol=0.0, max_iter=2)
        return plan.windowed, s

    def digest(t):  # every bit counts, without a second copy on the card
        return t.cpu().numpy().view(np.uint32)

    for call in (spmv, pagerank):
        on, out = call()
        assert on
        want = digest(out).copy()
        held = _fill(torch)
        on, out = call()
        assert not on
        np.testing.assert_array_equal(digest(out), want)
        del held
        torch.cuda.empty_cache()
        on, out = call()  # and with the memory back
        assert on
        np.testing.assert_array_equal(digest(out), want)
    # the backward's transpose alone needs more than FREE: a clean error, then the plan
    held = _fill(torch)
    with pytest.raises(Exception, match="GD_ERR_ALLOC"):
        backward()
    del held
    torch.cuda.empty_cache()
    on, out = backward()
    assert on
    row = torch.repeat_interleave(torch.arange(m, device=device), torch.diff(off.long()))
    assert bool((out == gr[row] * x[col.long()]).all())
