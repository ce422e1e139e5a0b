"""The device CSR build with long runs of self-loops inside a row: the record
after a run is a duplicate exactly if it equals the last one before the run
(unsorted), however many loops, and how many 1024-record wavefronts, lie
between.  The host builder is the reference."""
import numpy as np
import pytest

from gardenia_ocl_amd import graph

pytestmark = pytest.mark.gpu


def _edges(kind, run, m):
    v = m // 2
    loops = [(v, v)] * run
    if kind == "same":       # equal records around every run
        e = [(v, m - 1)] + loops + [(v, m - 1)] + loops + [(v, m - 1), (v, 0)]
    elif kind == "other":    # different ones, then a twin next to its twin
        e = [(v, 0)] + loops + [(v, m - 1), (v, m - 1)] + loops + [(v, 0)]
    elif kind == "first":    # the row, and the list, start with loops
        e = loops + [(v, 0)] + loops + [(v, 0), (v, m - 1)]
    elif kind == "rows":     # loops end one row and start the next
        e = [(v, 0)] + loops + [(v + 1, v + 1)] * run + [(v + 1, 0)] + [(v + 2, 0), (v + 2, v + 2),
                                                                        (v + 2, 0)]
    else:                    # nothing but loops, then an edge of another row
        e = loops + [(v + 1, v)]
    return np.array(e, np.int32).T.copy()


@pytest.mark.parametrize("run", [1, 63, 64, 1021, 1022, 1023, 1024, 1025, 2047, 3072, 5001, 20000])
@pytest.mark.parametrize("kind", ["same", "other", "first", "rows", "only"])
@pytest.mark.parametrize("srt", [False, True])
def test_runs_of_self_loops(device, run, kind, srt):
    import torch

    m = 9
    src, dst = _edges(kind, run, m)
    for flags in ({}, {"remove_selfloops": False}, {"remove_redundents": False}):
        h = graph.csr_from_edges(m, src, dst, sorted=srt, **flags)
        d = graph.csr_from_edges_device(m, torch.from_numpy(src).to(device),
                                        torch.from_numpy(dst).to(device), sorted=srt, **flags)
        for name in ("row_offsets", "column_indices", "degree"):
            np.testing.assert_array_equal(d[name].cpu().numpy(), getattr(h, name), err_msg=str(flags))
