"""The batched-PPR search starts from the plan's defaults and can return them."""
import json

import numpy as np
import pytest

from gardenia_ocl_amd import autotune


def test_ppr_space_starts_from_the_defaults():
    assert {n: v[0] for n, v in autotune.PPR_SPACE.items()} == {
        "k_chunk": 0, "hub_cols": 32, "relabel": True}
    assert autotune.ppr_space(1 << 20, 256)["k_chunk"] == [0, 256, 128, 64]
    assert autotune.ppr_space(1 << 20, 192)["k_chunk"] == [0, 64]
    assert autotune.ppr_space(1 << 13, 128)["k_chunk"] == [128, 64]      # 4 MB of contributions
    assert autotune.ppr_space((1 << 13) + 1, 128)["k_chunk"] == [0, 128, 64]
    assert autotune.ppr_space(4, 64, {"k_chunk": [0, 256], "hub_cols": [16]}) == {
        "k_chunk": [0], "hub_cols": [16]}


@pytest.mark.gpu
def test_tuned_ppr_is_no_slower_choice_than_the_defaults(device):
    import torch

    from gardenia_ocl_amd import PersonalizedPageRankPlan, graph

    out_csr, in_csr = graph.rmat(13, 8, seed=3)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).to(device)  # noqa: E731
    args = t(in_csr.row_offsets), t(in_csr.column_indices), t(out_csr.degree)
    best, timings = autotune.tune_ppr(*args, 192, iters=1, repeats=1)
    defaults = {"k_chunk": 0, "hub_cols": 32, "relabel": True}
    assert timings[json.dumps(best, sort_keys=True)] <= timings[json.dumps(defaults, sort_keys=True)]
    info = PersonalizedPageRankPlan(*args, 192, relabel=True).info()
    assert info["k_chunk"] == 32 and info["hub_cols"] == 32  # what the defaults stand for
