"""What the engine is timed on: single calls of the step function (`LLM.step`), the call that everything the engine does
goes through, from one request's next token to a full portion of prompts beside decoding requests.

A case names a model, a precision, how many requests decode and how long their contexts are, and how many prompts of how
many tokens are run in the same step. The model's weights are random and always the same ones (a checkpoint, as a serving
process has it loaded, together with its cache and its captured steps); contexts, prompts and the decoded tokens come from
the seed. The requests that decode move on by one token a pass, as they do in use, and start over at the case's own
context after `ROOM` tokens; prompts are new requests in every pass.

The spread of the weights, the scale of the embedding and the factor on what a sub-layer adds are such that a rounding is not
blown up from layer to layer (a few tenths of a percent of the logits in bfloat16), as in trained models; with wilder ones two
correct computations would differ by more than a wrong one. No time depends on them.

Qwen2 models have the layer sizes that bench.py measures, the other decoders the groups of layers that it measures at the
width of 1,024 or 2,048, with dense feed-forwards throughout: where two scores of a router all but tie, two correct
computations take different experts, and no tolerance bounds what follows. A step returns the logits of the rows that were
asked for: every decoding request's, and each prompt's last.
"""

import math
from statistics import NormalDist

import numpy as np
import torch

WEIGHTS_SEED = 0
PORTION = 2048           # tokens of the steps that bring a context into the cache
ROOM = 4096              # decoded tokens after which a request starts over

QWEN2 = {"architectures": ["Qwen2ForCausalLM"], "head_dim": 128, "rope_theta": 1000000.0, "use_sliding_window": False,
         "hidden_act": "silu", "rms_norm_eps": 1e-6, "max_position_embeddings": 32768}
# tokens: the cache's size, for four times the largest case of the model
SIZES = {
    "qwen2-1.5b": dict(tokens=1 << 21, num_hidden_layers=28, hidden_size=1536, num_attention_heads=12, num_key_value_heads=2,
                       intermediate_size=8960, vocab_size=151936, tie_word_embeddings=True),
    "qwen2-7b": dict(tokens=1 << 19, num_hidden_layers=28, hidden_size=3584, num_attention_heads=28, num_key_value_heads=4,
                     intermediate_size=18944, vocab_size=152064, tie_word_embeddings=False),
    "dufelix-w1024": dict(tokens=1 << 19, width=1024, layers=8, heads=8, kv_heads=2, ff=4096, window=1024),
    "dufelix-w2048": dict(tokens=1 << 19, width=2048, layers=16, heads=16, kv_heads=4, ff=8192, window=1024),
    "netovik-w1024": dict(tokens=1 << 19, width=1024, layers=8, heads=8, kv_heads=2, ff=4096, window=1024),
    "netovik-w2048": dict(tokens=1 << 19, width=2048, layers=16, heads=16, kv_heads=4, ff=8192, window=1024),
    "mepapel-w1024": dict(tokens=1 << 19, width=1024, layers=8, heads=8, kv_heads=2, ff=4096, window=1024),
    "mepapel-w2048": dict(tokens=1 << 19, width=2048, layers=16, heads=16, kv_heads=4, ff=8192, window=1024),
}
VOCAB = 32768            # of the decoders other than Qwen2
HEAD = 128               # their head size


def case(model, dtype, decode=0, context=0, prompts=0, length=0):
    return {"model": model, "dtype": dtype, "decode": decode, "context": context, "prompts": prompts, "length": length}


def listed():
    cases = {
        # one user alone: the shortest step there is, where launches and the trips between kernels count
        "one-request": case("qwen2-1.5b", "bf16", decode=1, context=500),
        # the benchmark's own decode step
        "decode-8": case("qwen2-1.5b", "bf16", decode=8, context=2048),
        # a full decode batch: half weights, half cache
        "decode-64": case("qwen2-1.5b", "bf16", decode=64, context=2048),
        # a long document behind few requests
        "long-context": case("qwen2-1.5b", "bf16", decode=4, context=16000),
        # the benchmark's own prompt: one full portion
        "prompt-2048": case("qwen2-1.5b", "bf16", prompts=1, length=2048),
        # an ordinary question
        "prompt-300": case("qwen2-1.5b", "bf16", prompts=1, length=301),
        # a serving step at the token budget: portions of prompts beside requests that decode, in a larger model
        "serving-7b": case("qwen2-7b", "bf16", decode=24, context=1000, prompts=3, length=667),
        # the 32-bit path, decoding
        "decode-8-fp32": case("qwen2-1.5b", "fp32", decode=8, context=1000),
        # decoders with other mixers, decoding: latent attention, state spaces, gated heads
        "dufelix-decode-16": case("dufelix-w2048", "bf16", decode=16, context=1500),
        # prompts of odd lengths: time mixing, heads that see each other's scores, averages over the depth
        "netovik-prompts": case("netovik-w2048", "bf16", prompts=2, length=901),
        # a step of portions and single tokens in a small model: delta rule, state spaces, chunked attention, retention
        "mepapel-mixed": case("mepapel-w1024", "bf16", decode=12, context=700, prompts=2, length=450),
        # portions and single tokens in 32 bits
        "dufelix-mixed-fp32": case("dufelix-w1024", "fp32", decode=5, context=600, prompts=1, length=200),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def log_uniform(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompts", "mixed", "fp32", "design", "design", "design"])
    if kind == "decode":
        batch = log_uniform(rng, 1, 64)
        return case("qwen2-1.5b", "bf16", decode=batch, context=log_uniform(rng, 100, min(16000, 131072 // batch)))
    if kind == "prompts":
        prompts = rng.randint(1, 4)
        return case("qwen2-1.5b", "bf16", prompts=prompts, length=log_uniform(rng, 20, 2048 // prompts))
    if kind == "mixed":
        prompts = rng.randint(1, 3)
        return case("qwen2-7b", "bf16", decode=log_uniform(rng, 1, 24), context=log_uniform(rng, 100, 1000),
                    prompts=prompts, length=log_uniform(rng, 50, 2000 // prompts))
    if kind == "fp32":
        if rng.random() < 0.6:
            return case("qwen2-1.5b", "fp32", decode=log_uniform(rng, 1, 32), context=log_uniform(rng, 100, 1500))
        return case("dufelix-w1024", "fp32", decode=log_uniform(rng, 1, 16), context=log_uniform(rng, 100, 1000),
                    prompts=rng.randint(1, 2), length=log_uniform(rng, 20, 300))
    model = "%s-w%d" % (rng.choice(["dufelix", "netovik", "mepapel"]), rng.choice([1024, 2048]))
    c = case(model, "bf16")
    what = rng.choice(["decode", "prompts", "mixed"])
    if what != "prompts":
        c.update(decode=log_uniform(rng, 1, 32), context=log_uniform(rng, 100, 1500))
    if what != "decode":
        prompts = rng.randint(1, 3)
        c.update(prompts=prompts, length=log_uniform(rng, 20, 1800 // prompts))
    return c


# ---- the models

def groups(model):
    """The layers of the decoders other than Qwen2: groups of four, as bench.py describes them."""
    design, z = model.split("-")[0], SIZES[model]
    C, H, G, layers = z["width"], z["heads"], z["kv_heads"], []
    stretch = {"factor": 8.0, "original": 1024, "fast": 32.0, "slow": 1.0}
    for i in range(z["layers"]):
        mlp = {"kind": "dense", "ff": z["ff"]}
        state_space = {"heads": 2 * C // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}
        heads = {"heads": H, "kv_heads": G, "dim": HEAD, "vdim": HEAD, "scale": HEAD ** -0.5}
        if design == "dufelix":
            if i % 4 == 1:
                kind, mixer = "mamba2", state_space
            elif i % 4 == 3:
                kind, mixer = "attention", dict(heads, rot={"base": 10000.0, "dims": HEAD // 2, "scaling": stretch})
            else:
                kind = "latent_attention"
                mixer = {"heads": H, "dim": HEAD, "rot_dim": 64, "vdim": HEAD, "kv_rank": 192, "q_rank": 3 * C // 8,
                         "scale": (HEAD + 64) ** -0.5, "rot": {"base": 10000.0, "dims": 64, "scaling": stretch}}
        elif design == "netovik":
            if i % 4 == 2:
                kind = "attention"
                mixer = dict(heads, softcap=30.0, bias_max=512, bias_rows=32, mask={"size": z["window"], "keep_first": 64})
            else:
                kind, mixer = "wkv", {"heads": C // 64, "dim": 64, "rank": C // 32}
        else:
            mlp["limit"] = 7.0
            if i % 4 == 0:
                kind, half = "parallel", H // 2
                mixer = {"left": dict(heads, conv=4, mask={"size": z["window"]}, rot={"base": 500000.0, "dims": HEAD}),
                         "right": {"heads": half, "dim": HEAD, "vdim": HEAD, "rot": {"base": 10000.0, "dims": HEAD},
                                   "decay": [1.0 - 2.0 ** -(5 + 3 * h / (half - 1)) for h in range(half)]}}
            elif i % 4 == 1:
                kind, mixer = "mamba2", state_space
            else:
                kind, mixer = "delta", {"heads": H, "kv_heads": H // 2, "dim": HEAD, "vdim": HEAD, "conv": 4}
        layers.append({"type": kind, "mixer": mixer, "mlp": mlp})
    return layers


def config_of(model):
    z = SIZES[model]
    if model.startswith("qwen2"):
        return dict(QWEN2, **{k: v for k, v in z.items() if k != "tokens"})
    design = model.split("-")[0]
    config = {"architecture": design.capitalize(), "vocab": VOCAB, "width": z["width"], "norm": {"eps": 1e-6},
              "layers": groups(model)}
    config.update({"dufelix": {"embedding": {"scale": 8.0}}, "mepapel": {"residual_mult": 0.02},
                   "netovik": {"embedding": {"scale": 256.0}, "norm": {"eps": 1e-6, "groups": 4}}}[design])
    return config


def spread(model):
    """The weights' standard deviation."""
    return 0.01 if model.startswith("qwen2") else 0.02


def vocabulary(model):
    return SIZES[model].get("vocab_size", VOCAB)


_engine = {}             # the engine of the model at hand, as a serving process keeps it


def engine(model, dtype):
    if (model, dtype) not in _engine:
        from distie_amd import LLM

        for old in _engine.values():
            old.close()
        _engine.clear()
        torch.cuda.empty_cache()
        z = SIZES[model]
        _engine[model, dtype] = LLM(config=config_of(model), random_weights=True, seed=WEIGHTS_SEED, weights_std=spread(model),
                                    dtype=dtype, max_cache_tokens=z["tokens"], max_seqs=256, token_budget=PORTION,
                                    max_model_len=32768 if model.startswith("qwen2") else 8192)
    return _engine[model, dtype]


# ---- a case's requests

def contexts(case):
    """The tokens behind each decoding request: between three quarters of the case's context and all of it."""
    return [case["context"] - (37 * i) % max(1, case["context"] // 4) for i in range(case["decode"])]


def lengths(case):
    return [case["length"] - (13 * i) % max(1, case["length"] // 4) for i in range(case["prompts"])]


def tokens(case, seed):
    """-> (context of every decoding request, tokens decoded behind it, prompts)"""
    rng = np.random.default_rng([seed, case["decode"], case["context"], case["prompts"], case["length"]])
    vocab = vocabulary(case["model"])
    behind = [rng.integers(0, vocab, n).tolist() for n in contexts(case)]
    following = rng.integers(0, vocab, (ROOM, case["decode"])).tolist()
    return behind, following, [rng.integers(0, vocab, n).tolist() for n in lengths(case)]


class State:
    """The requests of a case in the engine's cache. They leave it with the state."""

    made = 0

    def __init__(self, case, seed):
        from distie_amd import StepEntry

        State.made += 1
        self.Entry = StepEntry
        self.llm = engine(case["model"], case["dtype"])
        self.behind, self.following, self.prompts = tokens(case, seed)
        self.decoding = ["s%d-%d" % (State.made, i) for i in range(case["decode"])]
        self.asked = ["s%d-prompt-%d" % (State.made, i) for i in range(case["prompts"])]
        self.begin()

    def begin(self):
        """The decoding requests' contexts, in portions."""
        step, room = [], PORTION
        for name, ids in zip(self.decoding, self.behind):
            self.llm.finish(name)
            while ids:
                step.append(self.Entry(name, ids[:room], []))
                ids, room = ids[room:], room - len(step[-1].tokens)
                if not room:
                    self.llm.step(step)
                    step, room = [], PORTION
        if step:
            self.llm.step(step)
        self.done = 0

    def __del__(self):
        for name in getattr(self, "decoding", ()):
            self.llm.finish(name)


def prepare(case, seed):
    return State(case, seed)


def run(state):
    if state.done == ROOM:
        state.begin()
    Entry, llm = state.Entry, state.llm
    step = [Entry(name, [token], [0]) for name, token in zip(state.decoding, state.following[state.done])]
    step += [Entry(name, ids, [len(ids) - 1]) for name, ids in zip(state.asked, state.prompts)]
    logits = llm.step(step)
    state.done += 1
    for name in state.asked:
        llm.finish(name)
    return logits


# ---- the same in 64 bits, in plain torch

F64 = torch.float64
GOLDEN, INTERVALS, MASK = 0x9E3779B97F4A7C15, 1 << 16, (1 << 64) - 1


class Weights:
    """The random weights by name: N(0, std) as a function of the seed, the name and the element (splitmix64, whose top 16
    bits choose an interval of the inverse distribution function and the next 24 a place in it), rounded to the precision
    the engine keeps them in. On "meta" they are counted and not made."""

    def __init__(self, model, dtype, device):
        self.device, self.kept, self.std = device, torch.bfloat16 if dtype == "bf16" else torch.float32, spread(model)
        self.seen, self.held = {}, {}
        if device != "meta":
            normal = NormalDist()
            end = normal.inv_cdf(2.0 ** -20)
            edges = [end] + [normal.inv_cdf(j / INTERVALS) for j in range(1, INTERVALS)] + [-end]
            edges = torch.tensor(edges, dtype=F64).to(torch.float32)
            self.lower, self.width = edges[:-1].to(device), (edges[1:] - edges[:-1]).to(device)

    @staticmethod
    def mix(x):
        x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & MASK
        x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & MASK
        return x ^ (x >> 31)

    def __call__(self, name, *shape):
        self.seen[name] = math.prod(shape)
        if self.device == "meta":
            return torch.empty(shape, dtype=F64, device="meta")
        if name not in self.held:
            self.held[name] = self.make(name, math.prod(shape)).view(shape)
        return self.held[name].to(F64)

    def make(self, name, count):
        key = 0xCBF29CE484222325
        for byte in name.encode():
            key = ((key ^ byte) * 0x100000001B3) & MASK
        base = self.mix(self.mix(WEIGHTS_SEED) ^ key)
        signed = lambda x: x - (1 << 64) if x >> 63 else x  # noqa: E731
        shift = lambda x, bits: (x >> bits) & ((1 << (64 - bits)) - 1)  # noqa: E731
        out = torch.empty(count, dtype=self.kept, device=self.device)
        for at in range(0, count, 1 << 26):
            n = min(1 << 26, count - at)
            x = torch.arange(at, at + n, dtype=torch.int64, device=self.device) * signed(GOLDEN) + signed(base)
            x = (x ^ shift(x, 30)) * signed(0xBF58476D1CE4E5B9)
            x = (x ^ shift(x, 27)) * signed(0x94D049BB133111EB)
            x = x ^ shift(x, 31)
            interval = shift(x, 48)
            place = (shift(x, 24) & 0xFFFFFF).to(torch.float32) * 2.0 ** -24
            out[at:at + n] = ((self.lower[interval] + self.width[interval] * place) * self.std).to(self.kept)
        return out


def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def silu(x):
    return x * torch.sigmoid(x)


def frequencies(rot):
    """-> (frequencies of the pairs, factor on cosine and sine)"""
    dims, base, s = rot["dims"], rot["base"], rot.get("scaling")
    f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    if s:                                                   # a ramp over the dimensions
        where = lambda turns: dims * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(where(s["fast"])), 0), min(math.ceil(where(s["slow"])), dims - 1)
        ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
        return [x / s["factor"] * r + x * (1 - r) for x, r in zip(f, ramp)], 0.1 * math.log(s["factor"]) + 1.0
    return f, 1.0


def turn(x, rot, neighbours=False):
    """x [B, T, heads, D]: the first dims of every head turned by the position."""
    if not rot:
        return x
    f, factor = frequencies(rot)
    angle = torch.arange(x.shape[1], dtype=F64, device=x.device)[:, None] * torch.tensor(f, dtype=F64, device=x.device)
    cos, sin = (angle.cos() * factor)[:, None, :], (angle.sin() * factor)[:, None, :]
    dims = rot["dims"]
    first, second = (slice(0, dims, 2), slice(1, dims, 2)) if neighbours else (slice(0, dims // 2), slice(dims // 2, dims))
    out = x.clone()
    out[..., first] = x[..., first] * cos - x[..., second] * sin
    out[..., second] = x[..., second] * cos + x[..., first] * sin
    return out


def seen_keys(T, mask, device, chunks=False):
    i, j = torch.arange(T, device=device)[:, None], torch.arange(T, device=device)[None, :]
    seen = j <= i
    if mask and chunks:
        seen = seen & (i // mask["size"] == j // mask["size"])
    elif mask:
        seen = seen & ((i - j < mask["size"]) | (j < mask.get("keep_first", 0)))
    return seen


def softmax(scores, seen, sink=None):
    """Over the keys that are seen; `sink`: one more term in the sum, without a key."""
    scores = scores.masked_fill(~seen, -math.inf)
    top = scores.max(-1, keepdim=True).values
    if sink is not None:
        top = torch.maximum(top, sink)
    e = torch.exp(scores - top)
    return e / (e.sum(-1, keepdim=True) + (torch.exp(sink - top) if sink is not None else 0.0))


def attend(q, k, v, scale, mask=None, sinks=None, chunks=False):
    """q [B, T, H, D], k [B, T, G, D], v [B, T, G, E] -> [B, T, H * E], head by head where all at once is too large."""
    B, T, H, _ = q.shape
    per, seen = H // k.shape[2], seen_keys(T, mask, q.device, chunks)
    at_once = max(1, min(per, (1 << 28) // (T * T)))
    out = torch.empty(B, T, H, v.shape[3], dtype=F64, device=q.device)
    for b in range(B):
        for h in range(0, H, at_once if per % at_once == 0 else 1):
            heads = slice(h, h + (at_once if per % at_once == 0 else 1))
            scores = torch.matmul(q[b, :, heads].transpose(0, 1).contiguous(), k[b, :, h // per].T) * scale
            weights = softmax(scores, seen, None if sinks is None else sinks[heads][:, None, None])
            out[b, :, heads] = torch.matmul(weights, v[b, :, h // per]).transpose(0, 1)
    return out.reshape(B, T, -1)


def short_conv(x, filters, bias=0.0):
    taps, T = filters.shape[1], x.shape[1]
    x = torch.cat([x.new_zeros(x.shape[0], taps - 1, x.shape[2]), x], 1)
    return sum(x[:, j:j + T] * filters[:, j] for j in range(taps)) + bias


def over_heads(x, heads):
    return x.repeat_interleave(heads // x.shape[2], 2)


def state_space(h, w, p, m, eps):
    B, T, C = h.shape
    H, P, N = m["heads"], m["vdim"], m["state"]
    inner = H * P
    z, xbc, dt = torch.split(h @ w(p + "in", 2 * inner + 2 * N + H, C).T, [inner, inner + 2 * N, H], -1)
    xbc = silu(short_conv(xbc, w(p + "conv", inner + 2 * N, m["conv"]), w(p + "conv.b", inner + 2 * N)))
    x, b, c = xbc[..., :inner].view(B, T, H, P), xbc[..., inner:inner + N], xbc[..., inner + N:]
    dt = torch.nn.functional.softplus(dt + w(p + "dt_bias", H), threshold=700)
    keep = torch.exp(-torch.exp(w(p + "A_log", H)) * dt)
    S, y = h.new_zeros(B, H, N, P), torch.empty_like(x)
    for t in range(T):
        S = keep[:, t, :, None, None] * S + b[:, t, None, :, None] * (dt[:, t, :, None] * x[:, t])[:, :, None, :]
        y[:, t] = torch.matmul(c[:, t, None, None, :], S)[:, :, 0]
    y = y + w(p + "D", H)[:, None] * x
    return rms(y.reshape(B, T, inner) * silu(z), eps) @ w(p + "o", C, inner).T


def latent_attention(h, w, p, m, eps):
    B, T, C = h.shape
    H, D, R, E, rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
    q = (rms(h @ w(p + "dq", m["q_rank"], C).T, eps) @ w(p + "uq", H * (D + R), m["q_rank"]).T).view(B, T, H, D + R)
    q = torch.cat([q[..., :D], turn(q[..., D:], m["rot"], True)], -1)
    down = h @ w(p + "dkv", rank + R, C).T
    latent = rms(down[..., :rank], eps)
    turned = turn(down[..., rank:].view(B, T, 1, R), m["rot"], True).expand(B, T, H, R)
    k = torch.cat([(latent @ w(p + "uk", H * D, rank).T).view(B, T, H, D), turned], -1)
    v = (latent @ w(p + "uv", H * E, rank).T).view(B, T, H, E)
    return attend(q, k, v, m["scale"], sinks=w(p + "sink", H)) @ w(p + "o", C, H * E).T


def gated_attention(h, w, p, m, eps):
    B, T, C = h.shape
    H, G, D, E = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q = turn((h @ w(p + "q", H * D, C).T).view(B, T, H, D), m["rot"])
    k = turn((h @ w(p + "k", G * D, C).T).view(B, T, G, D), m["rot"])
    o = attend(q, k, (h @ w(p + "v", G * E, C).T).view(B, T, G, E), m["scale"])
    gate = torch.sigmoid(h @ w(p + "g", H, C).T)
    return (o.view(B, T, H, E) * gate[..., None]).reshape(B, T, H * E) @ w(p + "o", C, H * E).T


def time_mixing(h, w, p, m, eps):
    B, T, C = h.shape
    H, D = m["heads"], m["dim"]
    before = torch.cat([torch.zeros_like(h[:, :1]), h[:, :-1]], 1)
    mixed = {n: h + (before - h) * w(p + "mu." + n, C) for n in "rkvgw"}
    r, k, v = ((mixed[n] @ w(p + n, H * D, C).T).view(B, T, H, D) for n in "rkv")
    gate = silu(mixed["g"] @ w(p + "g", H * D, C).T)
    decay = torch.tanh(mixed["w"] @ w(p + "w1", m["rank"], C).T) @ w(p + "w2", H * D, m["rank"]).T + w(p + "w0", H * D)
    decay, u = torch.exp(-torch.exp(decay)).view(B, T, H, D), w(p + "u", H, D)
    S, o = h.new_zeros(B, H, D, D), torch.empty_like(r)
    for t in range(T):
        pair = k[:, t, :, :, None] * v[:, t, :, None, :]
        o[:, t] = torch.matmul(r[:, t, :, None, :], S + u[:, :, None] * pair)[:, :, 0]
        S = decay[:, t, :, :, None] * S + pair
    return (rms(o, eps).reshape(B, T, H * D) * gate) @ w(p + "o", C, H * D).T


def mixed_heads(h, w, p, m, eps):
    B, T, C = h.shape
    H, G, D, rows, cap = m["heads"], m["kv_heads"], m["dim"], m["bias_rows"], m["softcap"]
    q = rms((h @ w(p + "q", H * D, C).T + w(p + "q.b", H * D)).view(B, T, H, D), eps)
    v = (h @ w(p + "k", G * D, C).T + w(p + "k.b", G * D)).view(B, T, G, D)
    k, half = rms(v, eps), rows // 2
    steps = math.log(m["bias_max"] / half)

    def row_of(n):
        if n < half:
            return n
        place = math.log(n / half) / steps * (rows - half)
        return min(rows - 1, half + math.floor(round(place) if abs(place - round(place)) < 1e-9 else place))

    by_distance = w(p + "rel", rows, H)[torch.tensor([row_of(n) for n in range(T)], device=h.device)]
    at = torch.arange(T, device=h.device)
    bias = by_distance[(at[:, None] - at[None, :]).clamp(min=0)].permute(2, 0, 1)
    seen, out = seen_keys(T, m["mask"], h.device), torch.empty(B, T, H, D, dtype=F64, device=h.device)
    for b in range(B):
        scores = torch.matmul(q[b].transpose(0, 1).contiguous(), over_heads(k, H)[b].permute(1, 2, 0).contiguous()) * m["scale"]
        scores = cap * torch.tanh(scores / cap) + bias      # (the mix of the heads is the identity in random weights)
        weights = softmax(scores, seen, torch.zeros((), dtype=F64, device=h.device))
        out[b] = torch.matmul(weights, over_heads(v, H)[b].transpose(0, 1).contiguous()).transpose(0, 1)
    return out.reshape(B, T, H * D) @ w(p + "o", C, H * D).T


def chunked_attention(h, w, p, m, eps):
    B, T, C = h.shape
    H, G, D, E = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    sizes = {"q": H * D, "k": G * D, "v": G * E}
    q, k, v = (short_conv(h @ w(p + n, s, C).T + w(p + n + ".b", s), w(p + n + ".conv", s, m["conv"])) for n, s in sizes.items())
    q, k = (turn(rms(x.view(B, T, -1, D), eps), m["rot"], True) for x in (q, k))
    o = attend(q, k, v.view(B, T, G, E), m["scale"], m["mask"], chunks=True)
    return o @ w(p + "o", C, H * E).T + w(p + "o.b", C)


def retention(h, w, p, m, eps):
    B, T, C = h.shape
    H, D, E = m["heads"], m["dim"], m["vdim"]
    q, k = (turn((h @ w(p + n, H * D, C).T).view(B, T, H, D), m["rot"]) for n in "qk")
    k, v = k * D ** -0.5, (h @ w(p + "v", H * E, C).T).view(B, T, H, E)
    keep = torch.tensor(m["decay"], dtype=F64, device=h.device)[:, None, None]
    S, o = h.new_zeros(B, H, D, E), torch.empty_like(v)
    for t in range(T):
        S = keep * S + k[:, t, :, :, None] * v[:, t, :, None, :]
        o[:, t] = torch.matmul(q[:, t, :, None, :], S)[:, :, 0]
    return (rms(o, eps).reshape(B, T, H * E) * silu(h @ w(p + "g", H * E, C).T)) @ w(p + "o", C, H * E).T


def delta_rule(h, w, p, m, eps):
    B, T, C = h.shape
    H, G, D, E = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    sizes = {"q": G * D, "k": G * D, "v": H * E}
    q, k, v = (silu(short_conv(h @ w(p + n, s, C).T, w(p + n + ".conv", s, m["conv"]))) for n, s in sizes.items())
    q, k = (x.view(B, T, G, D) for x in (q, k))
    q, k = (over_heads(x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6), H) for x in (q, k))
    q, v = q * D ** -0.5, v.view(B, T, H, E)
    beta = torch.sigmoid(h @ w(p + "b", H, C).T)
    step = torch.nn.functional.softplus(h @ w(p + "a", H, C).T + w(p + "dt_bias", H), threshold=700)
    keep = torch.exp(-torch.exp(w(p + "A_log", H)) * step)
    S, o = h.new_zeros(B, H, D, E), torch.empty_like(v)
    for t in range(T):
        S = keep[:, t, :, None, None] * S
        u = beta[:, t, :, None] * (v[:, t] - torch.matmul(k[:, t, :, None, :], S)[:, :, 0])
        S = S + k[:, t, :, :, None] * u[:, :, None, :]
        o[:, t] = torch.matmul(q[:, t, :, None, :], S)[:, :, 0]
    return (rms(o, eps).reshape(B, T, H * E) * silu(h @ w(p + "g", H * E, C).T)) @ w(p + "o", C, H * E).T


def side_by_side(h, w, p, m, eps):
    left, right = chunked_attention(h, w, p + "left.", m["left"], eps), retention(h, w, p + "right.", m["right"], eps)
    return 0.5 * (rms(left, eps) + rms(right, eps))


def dense(h, w, p, ff, act, limit=None):
    C = h.shape[-1]
    gate, up = h @ w(p + "gate", ff, C).T, h @ w(p + "up", ff, C).T
    if limit is not None:
        gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
        return (gate * torch.sigmoid(1.702 * gate) * (up + 1)) @ w(p + "down", C, ff).T
    return (act(gate) * up) @ w(p + "down", C, ff).T


def qwen2_rows(w, model, ids, rows):
    c = config_of(model)
    C, D, H, G, F, eps = (c[k] for k in ("hidden_size", "head_dim", "num_attention_heads", "num_key_value_heads",
                                         "intermediate_size", "rms_norm_eps"))
    embed = w("model.embed_tokens.weight", c["vocab_size"], C)
    x, rot = embed[ids], {"dims": D, "base": c["rope_theta"]}
    B, T = ids.shape
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = rms(x, eps)
        q, k, v = ((h @ w(f"{p}self_attn.{n}_proj.weight", s * D, C).T + w(f"{p}self_attn.{n}_proj.bias", s * D)).view(B, T, s, D)
                   for n, s in (("q", H), ("k", G), ("v", G)))
        x = x + attend(turn(q, rot), turn(k, rot), v, D ** -0.5) @ w(p + "self_attn.o_proj.weight", C, H * D).T
        h, gate, up, down = rms(x, eps), w(p + "mlp.gate_proj.weight", F, C), w(p + "mlp.up_proj.weight", F, C), \
            w(p + "mlp.down_proj.weight", C, F)
        for b in range(B):
            x[b] += (silu(h[b] @ gate.T) * (h[b] @ up.T)) @ down.T
    x = rms(x[torch.arange(B, device=ids.device), rows], eps)
    return x @ (embed if c["tie_word_embeddings"] else w("lm_head.weight", c["vocab_size"], C)).T


def design_rows(w, model, ids, rows):
    c, z, design = config_of(model), SIZES[model], model.split("-")[0]
    eps, C = c["norm"]["eps"], z["width"]
    embed = w("embed", VOCAB, C)
    B, T = ids.shape
    x = embed[ids] * c.get("embedding", {}).get("scale", 1.0)
    apart = (lambda y: rms(y.view(B, T, 4, C // 4), eps).reshape(B, T, C)) if design == "netovik" else (lambda y: rms(y, eps))
    mixers = {"mamba2": state_space, "latent_attention": latent_attention, "wkv": time_mixing, "delta": delta_rule,
              "parallel": side_by_side, "attention": mixed_heads if design == "netovik" else gated_attention}
    gelu = lambda y: torch.nn.functional.gelu(y, approximate="tanh")  # noqa: E731
    for i, layer in enumerate(c["layers"]):
        p, m, mlp, mult = f"l{i}.", layer["mixer"], layer["mlp"], c.get("residual_mult", 1.0)
        before = (lambda y: rms(y, eps)) if design == "dufelix" else (lambda y: y)
        y = mixers[layer["type"]](before(x), w, p + "mix.", m, eps)
        x = x + mult * apart(y)
        y = dense(before(x), w, p + "mlp.", mlp["ff"], gelu if design == "dufelix" else silu, mlp.get("limit"))
        x = x + mult * apart(y)          # (the average over the depth takes the last result alone in random weights)
    x = apart(x)[torch.arange(B, device=ids.device), rows]
    return x @ (embed if design == "netovik" else w("head", VOCAB, C)).T


def exact(case, seed):
    cost = sum(n * n for n in contexts(case) + lengths(case))
    if cost > 3e8:                                          # the scores of a long context in 64 bits
        return None
    w = Weights(case["model"], case["dtype"], "cuda")
    behind, following, prompts = tokens(case, seed)
    sequences = [ids + [token] for ids, token in zip(behind, following[0])] + prompts
    rows_of = qwen2_rows if case["model"].startswith("qwen2") else design_rows
    out = torch.empty(len(sequences), vocabulary(case["model"]), dtype=F64, device="cuda")
    order = sorted(range(len(sequences)), key=lambda i: len(sequences[i]))
    while order:                                            # requests of like length together, filled up behind their last token
        longest = len(sequences[order[-1]])
        part = order[-max(1, (1 << 15) // longest):]
        del order[-len(part):]
        ids = torch.zeros(len(part), longest, dtype=torch.int64)
        for row, i in enumerate(part):
            ids[row, :len(sequences[i])] = torch.tensor(sequences[i])
        last = torch.tensor([len(sequences[i]) - 1 for i in part])
        out[torch.tensor(part)] = rows_of(w, case["model"], ids.cuda(), last.cuda())
    return out


# ---- what a step cannot do without

def kept(case):
    """-> (elements a cached token takes in all layers, 32-bit elements of state a request has in all layers, flops of a query
    on one visible key in all layers, flops of a token on the states)"""
    c = config_of(case["model"])
    if case["model"].startswith("qwen2"):
        L, D = c["num_hidden_layers"], c["head_dim"]
        return 2 * L * c["num_key_value_heads"] * D, 0, 4 * L * c["num_attention_heads"] * D, 0
    paged = state = pair = own = 0
    for layer in c["layers"]:
        m = layer["mixer"]
        left = m.get("left", m)
        if layer["type"] == "latent_attention":
            paged += m["kv_rank"] + m["rot_dim"]
            pair += 2 * m["heads"] * (2 * m["kv_rank"] + m["rot_dim"])
        elif layer["type"] in ("attention", "parallel"):
            paged += left["kv_heads"] * left["dim"] * (1 if "softcap" in m else 2)
            pair += 4 * left["heads"] * left["dim"]
        elements = {"mamba2": lambda: m["heads"] * m["vdim"] * m["state"], "wkv": lambda: m["heads"] * m["dim"] ** 2,
                    "delta": lambda: m["heads"] * m["dim"] * m["vdim"],
                    "parallel": lambda: m["right"]["heads"] * m["right"]["dim"] * m["right"]["vdim"]}.get(layer["type"], int)()
        state += elements
        own += 6 * elements
    return paged, state, pair, own


def work(case):
    w = Weights(case["model"], case["dtype"], "meta")
    model, size = case["model"], 2 if case["dtype"] == "bf16" else 4
    one = torch.zeros(1, 1, dtype=torch.int64, device="meta")
    (qwen2_rows if model.startswith("qwen2") else design_rows)(w, model, one, one[0])
    c = config_of(model)
    rows, new = case["decode"] + case["prompts"], case["decode"] + sum(lengths(case))
    embed = w.seen["embed" if "embed" in w.seen else "model.embed_tokens.weight"]
    tied = c.get("tie_word_embeddings", not any(n in w.seen for n in ("head", "lm_head.weight")))
    head = embed
    body = sum(w.seen.values()) - embed - (0 if tied else head)
    window = SIZES[model].get("window", 1 << 30)
    paged, state, pair, own = kept(case)
    keys = sum(min(n + 1, window) for n in contexts(case))
    pairs = keys + sum(min(n, window) * n - min(n, window) ** 2 / 2 for n in lengths(case))
    out = rows * vocabulary(model) * 4
    moved = (body + head) * size + (keys + sum(lengths(case))) * paged * size + (2 * case["decode"] + case["prompts"]) * state * 4 + out
    return {"bytes": moved, "flops": 2 * body * new + 2 * head * rows + pairs * pair + own * new}


def tolerance(case):
    """Four times what products on other kernels, rounded or added up at other places, were seen to change."""
    return {"rel": 1e-5, "max": 1e-4} if case["dtype"] == "fp32" else {"rel": 0.03, "max": 0.2}
