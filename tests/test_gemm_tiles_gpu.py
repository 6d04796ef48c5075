"""The choice among tile kinds and parts of K for prompt-sized products: sizes at which each is taken, with edges in rows and columns."""
import math

import numpy as np
import pytest
import torch

from test_kernels_gpu import dev, rounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(129, 3584, 3584), (333, 3584, 18944), (511, 3590, 3584), (700, 2560, 2048), (450, 8192, 2048), (2047, 904, 4864),
                                   (900, 2048, 1536), (1400, 2560, 2048), (1100, 1030, 8192), (2047, 1152, 896), (257, 1536, 576)])
def test_products(ops16, M, N, K):
    """Plain bf16 and accumulated fp32 results, the latter finished at once and left for the norm, against 64 bits on the rounded operands."""
    rng = np.random.default_rng(M + N)
    bf = torch.bfloat16
    a, w, x = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (N, K), (M, N)))
    w /= math.sqrt(K)
    da, dw = dev(a, bf), dev(w, bf)
    want = dev(rounded(a, bf), torch.float64) @ dev(rounded(w, bf), torch.float64).t()
    # 32-bit sums of K products: an ulp of the sum of magnitudes (about 0.64 sqrt(K) here) for each of up to K additions in the worst case;
    # their signs are random, so that sqrt(K) of them is ample
    sums = 2.0 ** -24 * K * 0.8
    out = torch.empty((M, N), dtype=bf, device="cuda")
    ops16.gemm(da, dw, out)
    assert float((out.double() - want).abs().max()) <= sums + 2.0 ** -8 * float(want.abs().max())
    for defer in (False, True):
        acc = dev(x)
        ops16.gemm(da, dw, acc, accumulate=True, defer=defer)
        ops16.settle()
        assert float((acc.double() - want - dev(x, torch.float64)).abs().max()) <= sums + 2.0 ** -22


@pytest.mark.parametrize("M,F,K", [(2047, 4864, 896), (333, 1056, 512), (130, 18944, 256), (700, 8960, 192)])
def test_gate_and_up(ops16, M, F, K):
    """The gated product in every kind that pairs gate and up columns inside a block."""
    rng = np.random.default_rng(M + F)
    bf = torch.bfloat16
    a, wg, wu = (rng.standard_normal(s).astype(np.float32) for s in ((M, K), (F, K), (F, K)))
    wg, wu = wg / math.sqrt(K), wu / math.sqrt(K)
    out = torch.empty((M, F), dtype=bf, device="cuda")
    ops16.gemm(dev(a, bf), ops16.interleave_gate_up(dev(wg, bf), dev(wu, bf)), out, swiglu=True)
    z = dev(rounded(a, bf), torch.float64)
    g, u = z @ dev(rounded(wg, bf), torch.float64).t(), z @ dev(rounded(wu, bf), torch.float64).t()
    want = g / (1 + torch.exp(-g)) * u
    sums = 2.0 ** -24 * K * 0.8
    assert float((out.double() - want).abs().max()) <= 2 * sums * float(torch.maximum(g.abs(), u.abs()).max()) + 2.0 ** -8 * float(want.abs().max())
