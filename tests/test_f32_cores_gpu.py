"""The 32-bit product and attention on the matrix cores, at the edges of their tiles, runs of columns and chunks of keys."""
import math

import numpy as np
import pytest
import torch

import plain
from test_kernels_gpu import FakeStep, dev, ints, paged_setup

pytestmark = pytest.mark.gpu
ULP = 2.0 ** -24


@pytest.mark.parametrize("N,K", [(1, 4), (17, 132), (100, 1024), (33, 1028), (130, 2052), (300, 1536)])
def test_product(ops32, N, K):
    """Rows from one to several tiles, runs of 128 columns and groups of 1,024 whole and in part: against 64 bits, the same bits for a row
    in any batch, plain and accumulated into a strided output, finished at once and left for the norm that follows."""
    rng = np.random.default_rng(N * 7 + K)
    Ms = (1, 16, 17, 33, 64, 65, 129, 300)
    a, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((300, K), (N, K), (N,)))
    da, dw, db = dev(a), dev(w), dev(b)
    exact = a.astype(np.float64) @ w.astype(np.float64).T + b
    # a chain of 128 roundings, eight runs, the groups and the bias, each at most an ulp of the sum of magnitudes
    bound = (128 + 8 + K // 1024 + 3) * ULP * (np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64).T + np.abs(b) + 1)
    x = rng.standard_normal((300, N)).astype(np.float32)
    rows = acc_rows = None
    for M in reversed(Ms):
        out = torch.empty((M, N), device="cuda")
        ops32.gemm(da[:M], dw, out, bias=db)
        assert np.all(np.abs(out.cpu().numpy() - exact[:M]) <= bound[:M]), M
        wide = torch.zeros((M, N + 3), device="cuda")
        wide[:, :N] = dev(x[:M])
        ops32.gemm(da[:M], dw, wide[:, :N], bias=db, accumulate=True)
        assert np.all(np.abs(wide[:, :N].cpu().numpy() - (exact[:M] + x[:M])) <= bound[:M] + 4 * ULP * np.abs(x[:M])), M
        assert float(wide[:, N:].abs().max()) == 0.0
        left = dev(x[:M])
        ops32.gemm(da[:M], dw, left, bias=db, accumulate=True, defer=True)
        ops32.settle()
        if rows is None:
            rows, acc_rows = out, wide[:, :N].clone()
        assert torch.equal(out, rows[:M]) and torch.equal(wide[:, :N], acc_rows[:M]) and torch.equal(left, acc_rows[:M]), M


def test_product_with_infinities(ops32):
    """An infinity or a NaN stays in its own row or column; the columns that a run is filled up with add nothing."""
    a, w = torch.ones((70, 100), device="cuda"), torch.ones((40, 100), device="cuda")
    a[3, 99], w[5, 0] = math.inf, math.nan
    for M in (16, 70):
        out = torch.empty((M, 40), device="cuda")
        ops32.gemm(a[:M], w, out)
        want = torch.full((M, 40), 100.0, device="cuda")
        want[3], want[:, 5] = math.inf, math.nan
        assert torch.equal(torch.nan_to_num(out, nan=-1.0), torch.nan_to_num(want, nan=-1.0))


@pytest.mark.parametrize("H,G,D,page,window,chunk", [(4, 4, 32, 4, 0, 0), (14, 2, 64, 16, 0, 0), (16, 1, 96, 8, 130, 0), (6, 2, 128, 256, 0, 100),
                                                     (5, 5, 64, 16, 127, 0), (28, 4, 128, 16, 0, 0)])
def test_attention(ops32, H, G, D, page, window, chunk):
    """Requests whose lengths lie around the chunks of 128 keys, portions and single tokens: against 64 bits, and the same bits for a request
    alone (other cuts of the keys), with the keys walked by one wave, and with an infinite value behind the tokens that it concerns."""
    rng = np.random.default_rng(H * 100 + D + page)
    lengths, q_lens = [1, 127, 128, 129, 300], [1, 127, 3, 1, 40]
    ks, vs, cache, table = paged_setup(rng, lengths, G, D, page, torch.float32)
    qs, positions, slots, wants = [], [], [], []
    for s, (n, ql) in enumerate(zip(lengths, q_lens)):
        q_full = rng.standard_normal((n, H, D)).astype(np.float32)
        pos = np.arange(n)
        mask = plain.visible(n, window)
        if chunk:
            mask &= pos[:, None] // chunk == pos[None, :] // chunk
        k, v = ks[s].astype(np.float64), vs[s].astype(np.float64)
        full = np.empty((n, H, D))
        for h in range(H):
            sc = np.where(mask, q_full[:, h].astype(np.float64) @ k[:, h // (H // G)].T / math.sqrt(D), -np.inf)
            full[:, h] = plain.softmax(sc) @ v[:, h // (H // G)]
        qs.append(q_full[n - ql:])
        wants.append(full[n - ql:])
        positions += list(range(n - ql, n))
        slots += [s] * ql
    q, want = np.concatenate(qs).reshape(-1, H * D), np.concatenate(wants).reshape(-1, H * D)

    def run(first, n):
        out = torch.full((n, H * D), math.nan, device="cuda")
        step = FakeStep(ints(positions[first:first + n]), ints(slots[first:first + n]), table, None)
        ops32.paged_attention(dev(q[first:first + n]), H, G, D, cache, step, window, 1.0 / math.sqrt(D), out, mask_chunk=chunk)
        return out
    whole = run(0, len(q))
    # a score is off by D + 2 roundings of its terms' magnitudes (at most |q| |k| / sqrt(D)), a weight by that and a few ulp of the
    # exponential, an output by its weights' errors and 300 sums, all times the largest value
    score = (D + 2) * ULP * max(np.linalg.norm(x, axis=-1).max() for x in qs) * max(np.linalg.norm(k, axis=-1).max() for k in ks) / math.sqrt(D)
    bound = (2 * (score + 8 * ULP) + 310 * ULP) * max(np.abs(v).max() for v in vs)
    assert np.max(np.abs(whole.cpu().numpy() - want)) <= bound
    starts = np.cumsum([0] + q_lens)
    workspace = ops32.attn_workspace
    for s, ql in enumerate(q_lens):
        assert torch.equal(run(int(starts[s]), ql), whole[starts[s]:starts[s] + ql]), f"request {s} alone"
    try:
        ops32.attn_workspace = workspace[:16]
        assert torch.equal(run(0, len(q)), whole), "all keys walked by one wave"
    finally:
        ops32.attn_workspace = workspace
    # the last token's value of the request of 300 tokens: the tokens before it do not see it
    page_id = int(table[4, 299 // page])
    cache.v.view(-1, G * D, page)[page_id, :, 299 % page] = math.inf
    again = run(0, len(q))
    assert torch.equal(again[:-1], whole[:-1]) and not bool(torch.isfinite(again[-1]).any())
