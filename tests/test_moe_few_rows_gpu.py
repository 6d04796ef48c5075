"""The experts' products where an expert has few rows, at the edges of their panels of K and tiles, against 64 bits."""
import numpy as np
import pytest
import torch

import helpers

pytestmark = pytest.mark.gpu
BF16, F32 = 1, 0


@pytest.fixture(scope="module")
def ops():
    from hf_cpu_amd.kernels import ops as kernel_ops
    return kernel_ops.Ops(torch.bfloat16)


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 512, 1088, 2048, 2112])
def test_few_rows(ops, K, gated):
    """Experts of 0, 1, 31, 32 and 33 rows (one with two tiles), results of both types; 32-bit sums of exact products differ
    from 64 bits by at most K roundings of the sum of magnitudes."""
    rng = np.random.default_rng(K + gated)
    counts = [1, 31, 0, 33, 32]
    N, E, P = 192, len(counts), sum(counts)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int32)
    a = helpers.bf16_round(rng.standard_normal((P, K)).astype(np.float32))
    w = helpers.bf16_round(rng.standard_normal((E, N, K)).astype(np.float32))
    scale = rng.random(P).astype(np.float32)
    dev = lambda v, dt=None: torch.from_numpy(np.ascontiguousarray(v)).cuda().to(dt) if dt else torch.from_numpy(v).cuda()
    da, dw, ds, di = dev(a, torch.bfloat16), dev(w, torch.bfloat16), dev(scale), dev(ids)
    max_tiles = P // 32 + E
    row_pair = torch.empty(P, dtype=torch.int32, device="cuda")
    tiles = torch.empty(3 * max_tiles + 1, dtype=torch.int32, device="cuda")
    n_tiles = tiles[3 * max_tiles:]
    stream = torch.cuda.current_stream().cuda_stream
    assert ops.lib.hfa_moe_plan(di.data_ptr(), P, E, 32, row_pair.data_ptr(), tiles.data_ptr(), n_tiles.data_ptr(), stream) == 0
    sums = np.einsum("pk,pnk->pn", a.astype(np.float64), w[ids].astype(np.float64))
    size = np.einsum("pk,pnk->pn", np.abs(a).astype(np.float64), np.abs(w[ids]).astype(np.float64))
    bound = K * 2.0 ** -24 * size
    if gated:
        pairs = lambda v: (v.reshape(P, N // 64, 2, 32)[:, :, 0].reshape(P, N // 2), v.reshape(P, N // 64, 2, 32)[:, :, 1].reshape(P, N // 2))
        (g, u), (bg, bu) = pairs(sums * scale[:, None]), pairs(bound * scale[:, None])
        s = 1 / (1 + np.exp(-g))
        want = g * s * u
        # silu's slope is at most 1.1; the products' own roundings, the exponential's among them, are a few of the result's
        bound = 1.1 * bg * (np.abs(u) + bu) + np.abs(g * s) * bu + 2.0 ** -20 * np.abs(want)
    else:
        want = sums * scale[:, None]
        bound = bound * scale[:, None] + 2.0 ** -23 * np.abs(want)
    cols = N // 2 if gated else N
    for code, dt in ((F32, torch.float32), (BF16, torch.bfloat16)):
        out = torch.full((P + 1, cols), float("nan"), dtype=dt, device="cuda")
        assert ops.lib.hfa_moe_gemm(da.data_ptr(), K, BF16, 1, dw.data_ptr(), BF16, row_pair.data_ptr(), tiles.data_ptr(), n_tiles.data_ptr(),
                                    max_tiles, 32, out.data_ptr(), cols, code, 1, ds.data_ptr(), 0, N, K, 0, int(gated), 1.0, 0.0, 0.0,
                                    stream) == 0
        got = out.float().cpu().numpy().astype(np.float64)
        assert np.isnan(got[P]).all()
        err = np.abs(got[:P] - want) - (bound if code == F32 else bound + 2.0 ** -8 * (np.abs(want) + bound))
        assert err.max() <= 0, f"{err.max():.3e}"
