"""The best k of rows that are cut into slices, against the kernel that takes a row in one block and against numpy."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [10240, 10241, 20483, 151936])
@pytest.mark.parametrize("k", [1, 40, 256, 257])
def test_same_as_whole_rows(ops32, V, k):
    """One slice and several, k up to the most and beyond; rows in random order, ascending and descending, with ties by the dozen and by
    the thousand, all equal, with infinities, with NaNs, and all best values in one slice."""
    rng = np.random.default_rng(V + k)
    x = rng.standard_normal((12, V)).astype(np.float32)
    x[1].sort()
    x[2] = np.sort(x[2])[::-1]
    x[3] = np.round(x[3] * 200) / 200
    x[4] = np.round(x[4])
    x[5] = 0.25
    x[6, ::7], x[6, 3] = -math.inf, math.inf
    x[7] = -math.inf
    x[7, 5:5 + k // 2] = 1.0
    x[8, rng.integers(0, V, V // 3)] = math.nan
    x[9, V - 300:] += 10.0
    x[10] = np.where(rng.random(V) < 0.5, 0.0, -0.0)
    x[11] = math.nan
    logits = torch.from_numpy(x).cuda()
    ids, vals, none = ops32.topk(logits, k, want_stats=False)
    want_ids, want_vals, _ = ops32.topk(logits, k)
    assert none is None and torch.equal(ids, want_ids)
    assert torch.equal(torch.nan_to_num(vals, nan=7.0), torch.nan_to_num(want_vals, nan=7.0))
    for r in (0, 1, 2, 3, 4, 5, 6, 9, 10):
        order = np.argsort(-x[r], kind="stable")[:k]
        assert np.array_equal(ids[r].cpu().numpy(), order), r
    workspace = ops32.workspace
    try:
        ops32.workspace = workspace[:64]                     # too little for the slices' candidates
        assert torch.equal(ops32.topk(logits, k, want_stats=False)[0], want_ids)
    finally:
        ops32.workspace = workspace
