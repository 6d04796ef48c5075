"""What this engine is timed on: passes through its public entry points (``Session``, ``Engine.step`` and
``truncate``/``release``, ``Sampler.sample``) over the sizes that it is used with.

A case names its kind:

* ``decode``: one step in which each of ``batch`` requests brings one token; the requests hold between ``lo`` and ``hi`` tokens
  (their lengths spread evenly over the logarithm). The step's tokens are taken back afterwards (``truncate``), as a draft's are.
* ``prefill``: one prompt's next ``tokens`` tokens in one step behind ``past`` tokens that the cache holds, logits for its last.
* ``serve``: one step of a serving loop: two prompt portions (a new prompt of ``tokens``, the rest of another) beside ``batch``
  decoded tokens.
* ``turn``: ``batch`` prompts of ``lo`` to ``hi`` tokens in one step, ``steps`` decode steps with given tokens, and the requests
  are released: designs that keep a state, which cannot be wound back, go through whole turns.
* ``sample``: the next token of ``batch`` rows of logits, with the sampler's parameters.

Weights are random and made on the device from the seed by the engine's own rule (``Session`` with a configuration); their
sizes are those of the benchmark's shapes (``bench.py``, ``bench_design.py``) and of the single-layer tests (1.5B, 3B).
"""
import math

import numpy as np
import torch

import hf_cpu_amd
from hf_cpu_amd.kernels import Ops
from hf_cpu_amd.model import Model
from hf_cpu_amd.sampling import Sampler, SamplerParams
from hf_cpu_amd.sampling.rng import Rng
from hf_cpu_amd.session import Session


# ---- the models ---------------------------------------------------------------------------

def _qwen2(layers, hidden, heads, kv_heads, head_dim, ff, vocab, tied):
    return dict(architectures=["Qwen2ForCausalLM"], model_type="qwen2", num_hidden_layers=layers, hidden_size=hidden,
                num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=head_dim, intermediate_size=ff, vocab_size=vocab,
                rope_theta=1000000.0, rms_norm_eps=1e-6, tie_word_embeddings=tied, use_sliding_window=False,
                max_position_embeddings=32768, hidden_act="silu")


QWEN2 = {"0.5b": _qwen2(24, 896, 14, 2, 64, 4864, 151936, True), "1.5b": _qwen2(28, 1536, 12, 2, 128, 8960, 151936, True),
         "3b": _qwen2(36, 2048, 16, 2, 128, 11008, 151936, True), "7b": _qwen2(28, 3584, 28, 4, 128, 18944, 152064, False)}


GORIDRA_LAYERS = 4           # (half the benchmark's: every mixture layer is another chance of a tie between experts, see tolerance)


def _goridra():
    """Pairs of layers: keys and values of its own with a dense feed-forward, a reader of those with a mixture of experts."""
    def mixer(kv_from):
        m = dict(heads=16, kv_heads=4, dim=128, vdim=128, scale=1.0 / math.sqrt(128), rot=dict(dims=128, base=500000.0), mask=dict(size=1024))
        return m if kv_from is None else dict(m, kv_from=kv_from)
    moe = dict(kind="moe", expert=dict(ff=1024), router=dict(experts=32, top=4, groups=dict(count=4, keep=2)))
    layers = []
    for l in range(0, GORIDRA_LAYERS, 2):
        layers += [dict(type="attention", mixer=mixer(None), mlp=dict(kind="dense", ff=8192)), dict(type="attention", mixer=mixer(l), mlp=moe)]
    return dict(architecture="Goridra", vocab=32000, width=2048, logit_softcap=30.0, norm=dict(eps=1e-6), layers=layers)


def _mobupel():
    """Pairs of layers: attention with mixed heads beside the gated delta rule, with a dense feed-forward; a matrix memory with
    exponential gates."""
    left = dict(heads=16, kv_heads=4, dim=128, vdim=128, scale=1.0 / math.sqrt(128), conv=4)
    right = dict(heads=16, kv_heads=16, dim=128, vdim=128, conv=4, decay_rank=64, gate_rank=64)
    pair = [dict(type="parallel", mixer=dict(left=left, right=right), mlp=dict(kind="dense", ff=8192)),
            dict(type="mlstm", mixer=dict(heads=16, dim=128, vdim=128, gate_cap=15.0), mlp=None)]
    return dict(architecture="Mobupel", vocab=32000, width=2048, embedding=dict(scale=math.sqrt(2048)), logit_scale=1.0, norm=dict(eps=1e-6),
                layers=pair * 3)


def _shape(case):
    return {"goridra": _goridra, "mobupel": _mobupel}[case["model"]]() if case["model"] in ("goridra", "mobupel") else QWEN2[case["model"]]


# ---- the cases ----------------------------------------------------------------------------

def listed():
    return [
        # the smallest call: the next tokens of a full batch, drawn with the sampler's default parameters
        dict(name="sample-64", kind="sample", batch=64, vocab=151936, temp=0.8, top_k=40, top_p=0.95, min_p=0.05),
        # one conversation with the smallest model: a step is launches and their latencies
        dict(name="decode-1-0.5b", kind="decode", model="0.5b", dtype="bfloat16", batch=1, lo=300, hi=300),
        # the headline workload: 2,048-token prompts on the 7B shape, decoded at batch 1 and 8, and the prompt itself
        dict(name="decode-1-7b", kind="decode", model="7b", dtype="bfloat16", batch=1, lo=2060, hi=2060),
        dict(name="decode-8-7b", kind="decode", model="7b", dtype="bfloat16", batch=8, lo=2048, hi=2150),
        dict(name="prefill-2048-7b", kind="prefill", model="7b", dtype="bfloat16", tokens=2048, past=0),
        # a full decode batch of a server, requests of very different lengths
        dict(name="decode-64-7b", kind="decode", model="7b", dtype="bfloat16", batch=64, lo=64, hi=2048),
        # a follow-up question of odd length behind a conversation
        dict(name="prefill-333-7b", kind="prefill", model="7b", dtype="bfloat16", tokens=333, past=1024),
        # a step of continuous batching: prompt portions beside decoded tokens
        dict(name="serve-0.5b", kind="serve", model="0.5b", dtype="bfloat16", tokens=1500, batch=47, lo=40, hi=1900),
        # the 32-bit engine (--dtype float32), both directions
        dict(name="decode-8-fp32", kind="decode", model="0.5b", dtype="float32", batch=8, lo=100, hi=1000),
        dict(name="prefill-700-fp32", kind="prefill", model="0.5b", dtype="float32", tokens=700, past=0),
        # a mixture of experts, and a design with recurrences: prompts and the tokens after them
        dict(name="turn-goridra", kind="turn", model="goridra", dtype="bfloat16", batch=4, lo=300, hi=900, steps=4),
        dict(name="turn-mobupel", kind="turn", model="mobupel", dtype="bfloat16", batch=4, lo=300, hi=900, steps=4),
    ]


def draw(rng):
    """The same kinds over the whole range: sizes spread over their logarithm, so odd ones are the rule; long contexts and
    prompts go with few requests, and with small models where the listed cases' work would be exceeded."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "serve", "turn", "turn", "sample"])
    if kind == "sample":
        greedy, whole = rng.random() < 0.25, rng.random() < 0.15
        return dict(kind=kind, batch=size(1, 64), vocab=rng.choice([32000, 151936, 152064]), temp=0.0 if greedy else round(rng.uniform(0.5, 1.2), 2),
                    top_k=0 if whole else size(5, 200), top_p=round(rng.uniform(0.8, 1.0), 2), min_p=rng.choice([0.0, 0.05]))
    if kind == "turn":
        lo = size(20, 600)
        return dict(kind=kind, model=rng.choice(["goridra", "mobupel"]), dtype="bfloat16", batch=rng.randint(1, 4), lo=lo, hi=min(900, size(lo, 2 * lo)),
                    steps=rng.randint(1, 6))
    dtype = "float32" if rng.random() < 0.2 else "bfloat16"
    model = "0.5b" if dtype == "float32" else rng.choice(["0.5b", "1.5b", "3b", "7b", "7b"])
    if kind == "decode":
        batch = size(1, 64)
        lo = size(30, 1500)
        return dict(kind=kind, model=model, dtype=dtype, batch=batch, lo=lo, hi=size(lo, min(8192, max(2048 if batch < 16 else 1500, 8192 // batch))))
    if kind == "prefill":
        tokens = size(5, 700 if dtype == "float32" else 2048)
        past = 0 if rng.random() < 0.4 or tokens > 1500 else size(16, 1024 if tokens > 700 else 6000)
        return dict(kind=kind, model=model, dtype=dtype, tokens=tokens, past=0 if dtype == "float32" and past > 2000 else past)
    if dtype == "float32":
        return dict(kind=kind, model=model, dtype=dtype, tokens=size(30, 400), batch=size(2, 24), lo=40, hi=size(60, 600))
    return dict(kind=kind, model="0.5b" if model == "7b" else model, dtype=dtype, tokens=size(100, 1500), batch=size(4, 64), lo=40, hi=size(200, 1900))


def _lengths(case):
    """Tokens that each request of the case holds (or, in a turn, brings): from ``lo`` to ``hi`` over the logarithm, dealt so that
    neighbours differ."""
    n, lo, hi = case["batch"], case["lo"], case["hi"]
    even = [int(round(lo * (hi / lo) ** (i / max(n - 1, 1)))) for i in range(n)]
    step = next((s for s in (7, 5, 3, 11, 13) if math.gcd(s, n) == 1), 1)
    return [even[i * step % n] for i in range(n)]


SERVE_PAST, SERVE_REST = 300, 500                    # a serving step's second portion: the rest of a prompt that was begun before


def _requests(case, seed):
    """(requests: {id: tokens it holds before the pass}, entries of the pass: [(id, tokens, wanted places)])."""
    rng = np.random.default_rng(seed)
    vocab = _shape(case).get("vocab_size") or _shape(case)["vocab"]

    def toks(n):
        return [int(t) for t in rng.integers(0, vocab, n)]
    held, entries = {}, []
    if case["kind"] in ("decode", "serve"):
        for i, n in enumerate(_lengths(case)):
            held[f"d{i}"] = toks(n)
            entries.append((f"d{i}", toks(1), [0]))
    if case["kind"] == "serve":
        n = case["tokens"]
        rest = max(1, min(SERVE_REST, n // 3))
        held["rest"] = toks(SERVE_PAST)
        entries += [("rest", toks(rest), [rest - 1]), ("new", toks(n), [n - 1])]
    if case["kind"] == "prefill":
        n = case["tokens"]
        if case["past"]:
            held["p"] = toks(case["past"])
        entries.append(("p", toks(n), [n - 1]))
    if case["kind"] == "turn":                        # the prompts, and the tokens given to the decode steps
        entries = [(f"t{i}", toks(n), [n - 1]) for i, n in enumerate(_lengths(case))]
        held = {f"t{i}": toks(case["steps"]) for i in range(case["batch"])}
    return held, entries


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.kind = case["kind"]
    if s.kind == "sample":
        g = torch.Generator("cuda")
        g.manual_seed(seed)
        s.sampler = Sampler(Ops(torch.bfloat16))
        s.logits = torch.randn(case["batch"], case["vocab"], generator=g, device="cuda") * 1.5
        s.params = SamplerParams(case["temp"], case["top_k"], case["top_p"], case["min_p"]).check()
        s.seed = seed
        return s
    held, s.entries = _requests(case, seed)
    longest = max(len(held.get(r, ())) + len(t) for r, t, _ in s.entries)
    total = sum(len(t) + 32 for t in held.values()) + sum(len(t) + 32 for _, t, _ in s.entries)
    s.session = Session(hf_cpu_amd.config_from_dict(_shape(case)), dtype=case["dtype"], ctx_max=-(-(longest + 64) // 256) * 256, batch=2048,
                        page_size=16, max_seqs=len(s.entries) + 1, kv_tokens=total + 2048, seed=seed)
    eng = s.session.engine
    if s.kind == "turn":
        s.given = held
        return s
    # the requests' earlier tokens, in steps of 2,048 tokens as the scheduler would run them
    step, room = [], 2048
    for r, tokens in held.items():
        at = 0
        while at < len(tokens):
            n = min(room, len(tokens) - at)
            step.append((r, tokens[at:at + n], []))
            at, room = at + n, room - n
            if room == 0:
                eng.step(step)
                step, room = [], 2048
    if step:
        eng.step(step)
    s.back = [(r, len(held[r])) for r, _, _ in s.entries if r in held]
    s.new = [r for r, _, _ in s.entries if r not in held]
    if s.kind == "decode":                            # generation is under way: steps of this shape have run before
        for _ in range(2):
            run(s)
    return s


def run(s):
    if s.kind == "sample":
        wants = [(s.params, Rng(s.seed + i), 0) for i in range(s.logits.shape[0])]
        return np.array([c.token for c in s.sampler.sample(s.logits, wants)], dtype=np.int64)
    eng = s.session.engine
    if s.kind == "turn":
        out = [eng.step(s.entries).clone()]           # (the next step writes its logits to the same place)
        for k in range(len(s.given[s.entries[0][0]])):
            out.append(eng.step([(r, [s.given[r][k]], [0]) for r, _, _ in s.entries]).clone())
        for r, _, _ in s.entries:
            eng.release(r)
        return torch.stack(out)
    logits = eng.step(s.entries)
    for r, n in s.back:
        eng.truncate(r, n)
    for r in s.new:
        eng.release(r)
    return logits


# ---- what a pass cannot do without --------------------------------------------------------

def _tensor_sizes(case):
    """(weights a token's products use [elements], embedding and head apart; head elements)."""
    c = QWEN2[case["model"]]
    E, F, H, G, D, L = (c[k] for k in ("hidden_size", "intermediate_size", "num_attention_heads", "num_key_value_heads", "head_dim",
                                       "num_hidden_layers"))
    return L * (E * (H + 2 * G) * D + H * D * E + 3 * F * E), c["vocab_size"] * E


def _turn_work(case):
    """Goridra and Mobupel: every pass reads the weights it uses once (experts: those that its tokens choose), and the requests' keys,
    values and states (read and written)."""
    lengths, steps = _lengths(case), case["steps"]
    W, V, KV, T = 2048, 32000, 1024, sum(lengths)
    if case["model"] == "goridra":
        n = GORIDRA_LAYERS // 2
        dense = n * (W * (2048 + KV) + W * 2048) + n * (W * 2048 * 2) + n * (2 * 8192 * W + 32 * W)
        expert, moe_layers, attn_layers, state, mix = 2 * 1024 * W, n, 2 * n, 0, 4.0
    else:
        dense = 3 * (3 * W * W + (2 * 2048 + KV + 2048) * W + 4 * 2048 * W + (16 + 128) * W + 2 * 64 * 2048 + 2 * 8192 * W) + 3 * (5 * 2048 * W + 32 * W)
        expert, moe_layers, attn_layers, state, mix = 0, 0, 3, 3 * (16 * 128 * 128 + 16 * 128 * 129), 2.0 + 2.0 * 4
    flops = nbytes = 0.0
    for tokens, ctx in [(T, None)] + [(case["batch"], k) for k in range(steps)]:
        flops += 2.0 * tokens * (dense + moe_layers * 4 * expert) + 2.0 * case["batch"] * V * W + 5.0 * tokens * state
        nbytes += 2.0 * (dense + V * W + moe_layers * 32 * (1.0 - (1.0 - 4 / 32) ** tokens) * expert) + 4.0 * case["batch"] * V
        for n in lengths:
            seen = n * (n + 1) / 2 if ctx is None else n + ctx + 1
            flops += attn_layers * mix * 16 * 128 * seen
            nbytes += attn_layers * 2.0 * KV * (n if ctx is None else seen) + 2 * 4.0 * state
    return {"bytes": nbytes, "flops": flops}


def work(case):
    if case["kind"] == "sample":
        n = case["batch"] * case["vocab"]
        return {"bytes": 4.0 * n + 8.0 * case["batch"], "flops": 1.0 * n}
    if case["kind"] == "turn":
        return _turn_work(case)
    c, elem = QWEN2[case["model"]], 4 if case["dtype"] == "float32" else 2
    L, H, G, D, V = c["num_hidden_layers"], c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["vocab_size"]
    per_token, head = _tensor_sizes(case)
    held, entries = {}, []                            # (tokens held, tokens brought) a request
    if case["kind"] == "prefill":
        entries = [(case["past"], case["tokens"])]
    else:
        entries = [(n, 1) for n in _lengths(case)]
        if case["kind"] == "serve":
            entries += [(SERVE_PAST, max(1, min(SERVE_REST, case["tokens"] // 3))), (0, case["tokens"])]
    T, R = sum(n for _, n in entries), len(entries)
    pairs = sum(n * past + n * (n + 1) / 2 for past, n in entries)          # (query, key) pairs
    flops = 2.0 * T * per_token + 2.0 * R * head + L * 4.0 * H * D * pairs
    cache = L * 2.0 * G * D * elem * sum(past + 2 * n for past, n in entries)      # what was held is read, what is new written and read
    return {"bytes": elem * (per_token + head) + cache + 4.0 * R * V + elem * T * c["hidden_size"], "flops": flops}


def tolerance(case):
    """About four times what this engine's logits are off ``exact``'s (random weights let a rounding grow from layer to layer). Relative
    error and largest difference seen: 32 bits 4e-6, 2e-5; bf16 0.010, 0.06 (0.5b), 0.018 (1.5b), 0.027 (3b), 0.044, 0.23 (7b); Mobupel
    0.015, 0.14; Goridra 0.004, 0.02 where every choice of experts is the same, 0.03 where two experts' scores lie so close that a
    rounding to bf16 decides for one row (that row is off by 0.2, its largest difference by 0.9)."""
    if case["kind"] == "sample":
        return "exact"
    if case["dtype"] == "float32":
        return {"rel": 1.5e-5, "max": 1e-4}
    if case["kind"] == "turn":
        return {"rel": 0.1, "max": 0.95}
    if case["model"] == "0.5b":
        return {"rel": 0.04, "max": 0.25}
    return {"rel": 0.15, "max": 0.9}


# ---- the same in 64 bits ------------------------------------------------------------------

def _signed(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def _mix(z):
    """The finishing function of splitmix64 on int64 tensors (products wrap; shifts to the right fill with zeros)."""
    z = (z ^ ((z >> 30) & ((1 << 34) - 1))) * _signed(0xbf58476d1ce4e5b9)
    z = (z ^ ((z >> 27) & ((1 << 37) - 1))) * _signed(0x94d049bb133111eb)
    return z ^ ((z >> 31) & ((1 << 33) - 1))


def _random_tensor(seed, index, shape, rule, std, dtype):
    """Tensor ``index`` of a random model as 64-bit numbers: 16-bit fields of two words a value added up, scaled, rounded to the
    stored type."""
    n = int(np.prod(shape, dtype=np.int64))
    out = torch.empty(n, dtype=torch.float64, device="cuda")
    key = _mix(torch.tensor([_signed(seed * 0x9e3779b97f4a7c15 + index)], device="cuda"))
    scale = torch.tensor(np.float32(std / math.sqrt(8 * (65536.0 ** 2 - 1) / 12)), device="cuda")
    for at in range(0, n, 1 << 25):
        e = key + 2 * torch.arange(at, min(n, at + (1 << 25)), device="cuda")
        total = torch.zeros_like(e)
        for word in (_mix(e), _mix(e + 1)):
            for shift in (0, 16, 32, 48):
                total += (word >> shift) & 0xffff
        v = (total - 262140).float() * scale
        out[at:at + e.numel()] = ((1.0 + v) if rule == "one_plus_normal" else v).to(dtype).double()
    return out.view(*shape) if shape else out.view(())


class _Weights:
    """The model's tensors by name, each made when it is asked for (their order, sizes and spreads are the model's declaration)."""

    def __init__(self, case, seed):
        specs = [p for p in Model.from_config(hf_cpu_amd.config_from_dict(_shape(case))).param_specs() if not p.optional]
        self.specs = {p.name: (i, p) for i, p in enumerate(specs)}
        self.seed, self.dtype = seed, getattr(torch, case["dtype"])

    def __contains__(self, name):
        return name in self.specs

    def __getitem__(self, name):
        i, p = self.specs[name]
        return _random_tensor(self.seed, i, tuple(p.shape), p.init[0], p.init[1], self.dtype)


def _attend(q, k, v, scale, visible):
    """q [Tq, H, D], k and v [Tk, G, D]; ``visible(query rows)`` gives the mask over the keys."""
    Tq, H, _ = q.shape
    G, out = k.shape[1], torch.empty(Tq, H, v.shape[2], dtype=torch.float64, device="cuda")
    rows = max(1, (1 << 27) // (k.shape[0] * (H // G)))
    for g in range(G):
        heads = slice(g * (H // G), (g + 1) * (H // G))
        for at in range(0, Tq, rows):
            s = torch.matmul(q[at:at + rows, heads].transpose(0, 1).contiguous(), k[:, g].t().contiguous()) * scale
            s.masked_fill_(~visible(torch.arange(at, min(Tq, at + rows), device="cuda")), -math.inf)
            out[at:at + rows, heads] = torch.matmul(torch.softmax(s, dim=-1), v[:, g].contiguous()).transpose(0, 1)
    return out.reshape(Tq, -1)


def _angles(T, dims, base):
    i = torch.arange(dims // 2, dtype=torch.float64, device="cuda")
    t = torch.arange(T, dtype=torch.float64, device="cuda")[:, None] * base ** (-2.0 * i / dims)
    return torch.cos(t)[:, None, :], torch.sin(t)[:, None, :]


def _rotate_halves(v, base):
    c, s = _angles(v.shape[0], v.shape[2], base)
    a, b = v.chunk(2, dim=-1)
    return torch.cat([a * c - b * s, a * s + b * c], dim=-1)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _exact_qwen2(case, w, sequences, wanted):
    """Logits at the place ``wanted[i]`` of each whole sequence."""
    c = QWEN2[case["model"]]
    H, G, D, eps, base = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["rms_norm_eps"], c["rope_theta"]
    sizes = [len(t) for t in sequences]
    x = w["model.embed_tokens.weight"][torch.tensor(sum(sequences, []), device="cuda")]
    for l in range(c["num_hidden_layers"]):
        p = f"model.layers.{l}."
        h = _rms(x, w[p + "input_layernorm.weight"], eps)
        q, k, v = (h @ w[f"{p}self_attn.{n}_proj.weight"].t() + w[f"{p}self_attn.{n}_proj.bias"] for n in "qkv")
        att = []
        for qs, ks, vs in zip(q.split(sizes), k.split(sizes), v.split(sizes)):
            T = qs.shape[0]
            keys = torch.arange(T, device="cuda")
            att.append(_attend(_rotate_halves(qs.view(T, H, D), base), _rotate_halves(ks.view(T, G, D), base), vs.view(T, G, D),
                               1.0 / math.sqrt(D), lambda rows: keys[None, :] <= rows[:, None]))
        x = x + torch.cat(att) @ w[p + "self_attn.o_proj.weight"].t()
        h = _rms(x, w[p + "post_attention_layernorm.weight"], eps)
        m = torch.nn.functional.silu(h @ w[p + "mlp.gate_proj.weight"].t()).mul_(h @ w[p + "mlp.up_proj.weight"].t())
        x = x + m @ w[p + "mlp.down_proj.weight"].t()
    ends = torch.tensor(np.cumsum([0] + sizes[:-1]) + np.array(wanted), device="cuda")
    head = "lm_head.weight" if "lm_head.weight" in w else "model.embed_tokens.weight"
    return _rms(x[ends], w["model.norm.weight"], eps) @ w[head].t()


def _moe(h, w, p, ids, weights, expert):
    """Sum over a token's choices; ``expert(e, rows of h, their weights)`` gives an expert's weighted result."""
    out = torch.zeros_like(h)
    for e in range(int(ids.max()) + 1):
        row, at = torch.nonzero(ids == e, as_tuple=True)
        if row.numel():
            out.index_add_(0, row, expert(e, h[row], weights[row, at][:, None]))
    return out


def _exact_goridra(w, tokens):
    c = _goridra()
    eps, T = c["norm"]["eps"], len(tokens)
    x, kv = w["embed"][torch.tensor(tokens, device="cuda")], None
    keys = torch.arange(T, device="cuda")

    def norm(x, name):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], w[name], w[name + ".b"], eps)
    for l, lc in enumerate(c["layers"]):
        p, m, f = f"l{l}.", lc["mixer"], lc["mlp"]
        h = norm(x, p + "norm1")
        q = _rotate_halves((h @ w[p + "mix.q"].t()).view(T, 16, 128), m["rot"]["base"])
        if "kv_from" not in m:
            kv = (_rotate_halves((h @ w[p + "mix.k"].t()).view(T, 4, 128), m["rot"]["base"]), (h @ w[p + "mix.v"].t()).view(T, 4, 128))
        y = _attend(q, *kv, m["scale"], lambda rows: (keys[None, :] <= rows[:, None]) & (keys[None, :] // 1024 == rows[:, None] // 1024)) \
            @ w[p + "mix.o"].t()
        if f["kind"] == "dense":
            y = y + torch.nn.functional.gelu(h @ w[p + "mlp.up"].t()) @ w[p + "mlp.down"].t()
        else:
            s = torch.softmax(h @ w[p + "mlp.router"].t(), dim=-1)
            groups = s.view(T, 4, 8)
            kept = torch.zeros(T, 4, dtype=torch.bool, device="cuda").scatter_(1, groups.amax(-1).topk(2, dim=1).indices, True)
            best = groups.masked_fill(~kept[..., None], -1.0).view(T, 32).topk(4, dim=1)
            y = y + _moe(h, w, p, best.indices, best.values / (best.values.sum(-1, keepdim=True) + 1e-20), lambda e, a, s: s * (
                torch.relu(a @ w[f"{p}mlp.e{e}.up"].t()).square() @ w[f"{p}mlp.e{e}.down"].t()))
        x = x + y
    return c["logit_softcap"] * torch.tanh(norm(x, "final.norm") @ w["embed"].t() / c["logit_softcap"])


def _exact_mobupel(w, tokens):
    c = _mobupel()
    eps, T, W, H, G, D = c["norm"]["eps"], len(tokens), c["width"], 16, 4, 128
    silu, softplus, keys = torch.nn.functional.silu, torch.nn.functional.softplus, torch.arange(T, device="cuda")

    def conv(u, taps):
        padded = torch.cat([torch.zeros(3, u.shape[1], dtype=torch.float64, device="cuda"), u])
        return sum(padded[j:j + T] * taps[:, j] for j in range(4))

    def attention(h, p, m):
        """Softmax weights per head, mixed over the heads, applied to the values of each head's group."""
        q, k, v = (conv(h @ w[p + n].t(), w[f"{p}{n}.conv"]).view(T, -1, D) for n in "qkv")
        q, k = _rms(q, w[p + "q.norm"], eps), _rms(k, w[p + "k.norm"], eps)
        s = torch.matmul(q.transpose(0, 1).contiguous(), k.permute(1, 2, 0).repeat_interleave(H // G, dim=0).contiguous()) * m["scale"]
        s = torch.softmax(s.masked_fill(keys[None, :] > keys[:, None], -math.inf), dim=-1)
        mixed = (w[p + "talk"] @ s.view(H, T * T)).view(H, T, T)
        y = torch.matmul(mixed, v.transpose(0, 1).repeat_interleave(H // G, dim=0).contiguous())
        return (y.transpose(0, 1).reshape(T, -1) * torch.sigmoid(h @ w[p + "g"].t())) @ w[p + "o"].t()

    def delta(h, p):
        q, k, v = (silu(conv(h @ w[p + n].t(), w[f"{p}{n}.conv"])).view(T, H, D) for n in "qkv")
        q, k = (u / torch.sqrt((u * u).sum(-1, keepdim=True) + 1e-6) for u in (q, k))
        beta = torch.sigmoid(h @ w[p + "b"].t())[..., None]
        rate = torch.exp(w[p + "A_log"])[:, None]
        decay = torch.exp(-rate * softplus(h @ w[p + "a1"].t() @ w[p + "a2"].t() + w[p + "dt_bias"]).view(T, H, D))[..., None]
        S, o = torch.zeros(H, D, D, dtype=torch.float64, device="cuda"), torch.empty_like(v)
        for t in range(T):
            S = decay[t] * S
            u = beta[t] * (v[t] - (S * k[t][..., None]).sum(1))
            S = S + k[t][..., None] * u[:, None, :]
            o[t] = (S * q[t][..., None]).sum(1)
        o = _rms(o * D ** -0.5, w[p + "norm"], eps).view(T, -1)
        return (o * torch.sigmoid(h @ w[p + "g1"].t() @ w[p + "g2"].t())) @ w[p + "o"].t()

    def memory(h, p, m):
        q, k, v = ((h @ w[p + n].t()).view(T, H, D) for n in "qkv")
        cap = m["gate_cap"]
        log_i, z = (cap * torch.tanh((h @ w[p + n].t() + w[p + n + ".b"]) / cap) for n in "if")
        log_f = -softplus(-z)
        S = torch.zeros(H, D, D + 1, dtype=torch.float64, device="cuda")         # the last column: the normaliser
        most, o = torch.zeros(H, dtype=torch.float64, device="cuda"), torch.empty_like(v)
        v1 = torch.cat([v, torch.ones_like(v[..., :1])], dim=-1)
        for t in range(T):
            new = torch.maximum(log_f[t] + most, log_i[t])
            S = torch.exp(log_f[t] + most - new)[:, None, None] * S + (torch.exp(log_i[t] - new)[:, None] * k[t])[..., None] * v1[t][:, None, :]
            most = new
            y = (S * q[t][..., None]).sum(1) * D ** -0.5
            o[t] = y[:, :D] / (torch.maximum(y[:, D].abs(), torch.exp(-most)) + 1e-6)[:, None]
        return (_rms(o, 1.0, eps).view(T, -1) * w[p + "norm"] * torch.sigmoid(h @ w[p + "g"].t())) @ w[p + "o"].t()

    def sublayer(x, p, which, fn):
        h = _rms(x, w[p + "norm" + which], eps)
        return x + _rms(fn(h) * torch.sigmoid(h @ w[f"{p}rg{which}"].t() + w[f"{p}rg{which}.b"]), w[f"{p}norm{which}b"], eps)

    angle = keys[:, None].double() * 10000.0 ** (-2.0 * torch.arange(W // 2, dtype=torch.float64, device="cuda") / W)
    x = w["embed"][torch.tensor(tokens, device="cuda")] * c["embedding"]["scale"] + torch.stack([torch.sin(angle), torch.cos(angle)], dim=-1).view(T, W)
    for l, lc in enumerate(c["layers"]):
        p, m = f"l{l}.", lc["mixer"]
        if lc["type"] == "mlstm":
            x = sublayer(x, p, "1", lambda h: memory(h, p + "mix.", m))
        else:
            x = sublayer(x, p, "1", lambda h: 0.5 * (_rms(attention(h, p + "mix.left.", m["left"]), w[p + "mix.left.out"], eps)
                                                     + _rms(delta(h, p + "mix.right."), w[p + "mix.right.out"], eps)))
        if lc["mlp"] is not None:
            def feed_forward(h):
                z, (a, b, c3, e) = h @ w[p + "mlp.up"].t(), w[p + "mlp.act"]
                return (a * _rms(z, 1.0, eps) + b * _rms(z ** 2, 1.0, eps) + c3 * _rms(z ** 3, 1.0, eps) + e) @ w[p + "mlp.down"].t()
            x = sublayer(x, p, "2", feed_forward)
    return _rms(x, w["final.norm"], eps) @ w["head"].t()


def exact(case, seed):
    if case["kind"] == "sample":                      # (tokens: the draw is defined by its 32-bit operations)
        return None
    w = _Weights(case, seed)
    held, entries = _requests(case, seed)
    if case["kind"] == "turn":
        model = _exact_goridra if case["model"] == "goridra" else _exact_mobupel
        rows = [model(w, t + held[r])[len(t) - 1:] for r, t, _ in entries]
        return torch.stack(rows, dim=1)
    return _exact_qwen2(case, w, [held.get(r, []) + t for r, t, _ in entries], [len(held.get(r, [])) + n[0] for r, t, n in entries])
