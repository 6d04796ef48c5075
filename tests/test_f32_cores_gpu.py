"""The 32-bit product on the matrix cores, at the edges of its tiles and runs of columns."""
import math

import numpy as np
import pytest
import torch

from test_kernels_gpu import dev

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
