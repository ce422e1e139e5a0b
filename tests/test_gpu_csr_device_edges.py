"""The device CSR build at the edges of its passes: record counts around a
wavefront's 1024 records and a placement workgroup's 2048 edges, long runs of
self-loops and duplicates across those borders, one vertex, and a second
stream.  The host builder is the reference."""
import numpy as np
import pytest

from gardenia_ocl_amd import graph

pytestmark = pytest.mark.gpu


def _edges(kind, m, n, rng):
    src = rng.integers(0, m, n).astype(np.int32)
    dst = rng.integers(0, m, n).astype(np.int32)
    if kind == "loops":  # runs of self-loops between equal records of one row
        src[:] = m // 2
        dst[:] = m // 2
        dst[:: max(1, n // 5)] = m - 1
    elif kind == "dups":
        src[:] = np.repeat(rng.integers(0, m, n // 1500 + 1), 1500)[:n]
        dst[:] = (src + 1) % m
    elif kind == "last":  # empty rows before and after the only one in use
        src[:] = m // 3
    return src, dst


@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 2047, 2049, 4097, 70001])
@pytest.mark.parametrize("kind,srt,sym", [("random", True, False), ("loops", False, False),
                                          ("loops", True, True), ("dups", False, True),
                                          ("last", True, False)])
def test_build_at_pass_borders(device, n, kind, srt, sym):
    import torch

    rng = np.random.default_rng(n)
    for m in (1, 2, 777):
        src, dst = _edges(kind, m, n, rng)
        lo, hi = np.minimum(src, dst).astype(np.int64), np.maximum(src, dst).astype(np.int64)
        wt = ((lo * 131 + hi) % 1009).astype(np.float32) / 7.0
        h = graph.csr_from_edges(m, src, dst, wt, sorted=srt, symmetrize=sym)
        t = lambda a: torch.from_numpy(a).to(device)  # noqa: E731
        d = graph.csr_from_edges_device(m, t(src), t(dst), t(wt), sorted=srt, symmetrize=sym,
                                        stream=torch.cuda.Stream() if n % 2 else None)
        np.testing.assert_array_equal(d["row_offsets"].cpu().numpy(), h.row_offsets)
        np.testing.assert_array_equal(d["column_indices"].cpu().numpy(), h.column_indices)
        np.testing.assert_array_equal(d["degree"].cpu().numpy(), h.degree)
        np.testing.assert_array_equal(d["weight"].cpu().numpy(), h.weight)
