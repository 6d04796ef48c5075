"""Decoded tokens of requests whose lengths differ widely: the cuts of their keys."""
import math

import numpy as np
import pytest
import torch

import plain
from test_kernels_gpu import FakeStep, dev, ints, paged_setup, rounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,H,G,D,longest", [(40, 4, 2, 64, 1500), (130, 8, 4, 32, 900), (9, 7, 1, 128, 4096), (9, 2, 1, 96, 4101), (520, 2, 1, 32, 300)])
def test_ragged_batches(ops16, S, H, G, D, longest):
    """From one token to ``longest``: sixteen chunks, as many as 2,048 waves allow, a span at and beyond the 4,096 keys up to which a batch's
    keys are cut finer, and more than 512 tiles."""
    rng = np.random.default_rng(S + D)
    bf = torch.bfloat16
    lengths = [max(1, int(longest ** (i / (S - 1)))) for i in range(S)]
    lengths[-1] = longest
    ks, vs, cache, table = paged_setup(rng, lengths, G, D, 16, bf)
    q = rng.standard_normal((S, H, D)).astype(np.float32)
    want = np.empty((S, H * D))
    for s, n in enumerate(lengths):
        qf, k, v = rounded(q[s], bf), rounded(ks[s], bf), rounded(vs[s], bf)
        for h in range(H):
            w = plain.softmax(k[:, h // (H // G)] @ qf[h] / math.sqrt(D))
            want[s, h * D:(h + 1) * D] = w @ v[:, h // (H // G)]
    out = torch.empty((S, H * D), dtype=bf, device="cuda")
    step = FakeStep(ints([n - 1 for n in lengths]), ints(range(S)), table, None)
    ops16.paged_attention(dev(q.reshape(S, H * D), bf), H, G, D, cache, step, 0, 1.0 / math.sqrt(D), out)
    # probabilities and the output rounded to 8 bits of mantissa: half an ulp each of values up to the largest one (short requests)
    bound = 2.0 ** -8 * max(float(np.abs(v).max()) for v in vs)
    assert np.max(np.abs(out.float().cpu().numpy() - want)) <= bound
