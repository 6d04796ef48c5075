"""The recurrences' staging in pieces of four against their staging value by value (operands that no piece of four may be taken
from): the same values in the same places, so the same bits. The value-by-value results are checked elsewhere against whole sequences."""
import types

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
LENGTHS = [1, 16, 37, 15, 64]


@pytest.fixture(scope="module")
def ops():
    from hf_cpu_amd.kernels import ops as kernel_ops
    return kernel_ops.Ops(torch.float32)


def step():
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    return types.SimpleNamespace(q_start=ints([0] + list(np.cumsum(LENGTHS))), seq_slot=ints([3, 0, 4, 1, 2]), n_seqs=len(LENGTHS),
                                 max_q_len=max(LENGTHS), n_tokens=sum(LENGTHS))


def aside(t):
    """The same values in rows that start off every piece's boundary."""
    wide = torch.full((t.shape[0], t.shape[1] + 3), float("nan"), dtype=t.dtype, device=t.device)
    wide[:, 1:1 + t.shape[1]] = t
    return wide[:, 1:1 + t.shape[1]]


def both(run, state):
    out = []
    for place in (lambda t: t, aside):
        s = state.clone()
        y = run(place, s)
        again = run(place, s)                             # from the state just left
        out.append([y, again, s])
    for a, b in zip(*out):
        assert torch.equal(a, b) and torch.isfinite(a).all()


# (heads, key heads, key channels, columns): every number of lanes a column and values a lane, channels and columns that fill neither
SIZES = [(2, 1, 16, 64), (2, 2, 12, 5), (4, 2, 32, 33), (2, 1, 60, 32), (2, 2, 64, 16), (3, 1, 100, 48), (2, 1, 128, 16), (2, 2, 200, 17), (1, 1, 256, 16)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("gate", [0, 1, 2])
@pytest.mark.parametrize("H,G,N,P", SIZES)
def test_linear(ops, dtype, gate, H, G, N, P):
    g = torch.Generator(device="cuda").manual_seed(H + N + P)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, st = sum(LENGTHS), step()
    q, k, v = rand(T, G * N).to(dtype), rand(T, G * N).to(dtype), rand(T, H * P).to(dtype)
    z1, z2, bias, a_log, d = rand(T, H), rand(T, H), rand(H), rand(H) - 2, rand(H)
    floats = ops.scan_state_floats(H, N, P, normalizer=gate == 2)
    more = {0: dict(decay=torch.sigmoid(bias), skip=d), 1: dict(step_size=z1, step_bias=bias, a_log=a_log)}.get(gate)

    def run(place, s):
        y, denom = torch.empty(T, H * P, device="cuda"), torch.ones(T, H, device="cuda")
        kw = more or dict(exp_gates=(z1, z2, bias, d, 15.0), denom=denom)
        ops.linear_scan(place(q), place(k), place(v), G, N, H, P, s, st, y, q_scale=N ** -0.5, **kw)
        return torch.cat([y, denom], 1)
    both(run, torch.zeros(len(LENGTHS), floats + 2, device="cuda"))


@pytest.mark.parametrize("H,G,N,P", SIZES)
def test_delta(ops, H, G, N, P):
    g = torch.Generator(device="cuda").manual_seed(H + N + P)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, st = sum(LENGTHS), step()
    q, k, v, a, b = rand(T, G * N), rand(T, G * N), rand(T, H * P), rand(T, H * N), rand(T, H)
    dt_bias, a_log = rand(H * N), rand(H) - 1

    def run(place, s):
        y = torch.empty(T, H * P, device="cuda")
        ops.delta_scan(place(q), place(k), place(v), G, N, H, P, place(a), dt_bias, a_log, b, s, st, y, q_scale=N ** -0.5)
        return y
    both(run, torch.zeros(len(LENGTHS), ops.scan_state_floats(H, N, P), device="cuda"))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("H,G,N,P", SIZES)
def test_channels(ops, dtype, form, H, G, N, P):
    g = torch.Generator(device="cuda").manual_seed(H + N + P)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    T, st = sum(LENGTHS), step()
    q, k, v, z = rand(T, H * N).to(dtype), rand(T, H * N).to(dtype), rand(T, H * P).to(dtype), rand(T, H * N)
    lower = torch.rand(H * N, generator=g, device="cuda")

    def run(place, s):
        y = torch.empty(T, H * P, device="cuda")
        kw = dict(lower=lower, q_act="silu") if form == 0 else dict(tau=16.0)
        ops.channel_scan(place(q), None if form == 0 else place(k), place(v), H, N, P, z, None, s, st, y, q_scale=N ** -0.5, **kw)
        return y
    both(run, torch.zeros(len(LENGTHS), ops.scan_state_floats(H, N, P), device="cuda"))
