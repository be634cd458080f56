"""The work this framework is timed on: its matrix products, attention over a prompt, and decoders that
answer, from the smallest call to the longest context.

``listed()`` are the cases, ``draw(rng)`` gives one more of the same ranges.  A case's inputs come from a
seed alone (``prepare``), one pass goes through the public entry points (``run``), ``work`` is what a pass
cannot do without, and ``exact`` the same results in 64 bits without this package's code.

Decoders have random weights at the scales of a trained model's: projections N(0, 0.02), those that join
the stream smaller by the root of twice the layers, so that no layer drowns the stream.  Their output
matrix holds each token's embedding at the row of another token, its successor, so that every next token is
far ahead of the others: an answer is then the same for every correct order of the sums, and a wrong one
shows.
"""

from __future__ import annotations

import dataclasses
import math
from types import SimpleNamespace

import numpy as np
import torch

from iron_amd import kernels as K
from iron_amd.applications.llama import LLAMA_3_2_1B, Llama, Llama3RopeScaling, LlamaConfig
from iron_amd.applications.llama import shapes as llama_shapes
from iron_amd.applications.pufuzen import Pufuzen, PufuzenConfig
from iron_amd.applications.pufuzen import shapes as pufuzen_shapes
from iron_amd.lm import Entry, Sampler

BF16 = torch.bfloat16


# ---------------------------------------------------------------- the cases
def listed() -> list[dict]:
    return [
        # The smallest product: a narrow head over a few hundred rows, both matrices as a checkpoint stores them.
        dict(name="gemm 192x64x384", kind="gemm", m=192, n=64, k=384, b_col_maj=True, c_col_maj=True),
        # The product the framework is quoted on: B as the operator takes it by default.
        dict(name="gemm 2048", kind="gemm", m=2048, n=2048, k=2048, b_col_maj=False, c_col_maj=False),
        # A feed-forward's first product over a ragged prompt.
        dict(name="gemm 777x10240x2560", kind="gemm", m=777, n=10240, k=2560, b_col_maj=True, c_col_maj=False),
        # The largest product: many prompts' rows against a wide weight.
        dict(name="gemm 8192", kind="gemm", m=8192, n=8192, k=8192, b_col_maj=True, c_col_maj=False),
        # One row against a feed-forward's second matrix.
        dict(name="gemv 8192 to 2048", kind="gemv", m=2048, k=8192),
        # Causal attention of a ragged prompt, heads of 128.
        dict(name="attention 3001", kind="attention", heads=32, kv_heads=8, d=128, seq=3001, window=0),
        # A toy decoder's short answer: nothing but launches and the host.
        dict(name="toy answer", kind="answer", model="toy", context=256, history=0, turn=5, count=16, sampled=False),
        # A chat's first turn: a short question, a short answer.
        dict(name="1b answer 29+32", kind="answer", model="1b", context=2048, history=0, turn=29, count=32, sampled=False),
        # The usual one: a prompt of 512 tokens, drawn with temperature and top-k.
        dict(name="1b answer 512+64", kind="answer", model="1b", context=2048, history=0, turn=512, count=64, sampled=True),
        # A document read: what follows 7001 tokens (four portions, the last one ragged).
        dict(name="1b prompt 7001", kind="prompt", model="1b", context=8192, turn=7001),
        # A turn late in a long conversation: 12003 tokens held, 40 new ones, an answer.
        dict(name="1b turn behind 12003", kind="answer", model="1b", context=16384, history=12003, turn=40, count=24, sampled=False),
        # Eight requests of ragged lengths served as one batch by a hybrid, and the answers scored.
        dict(name="serve 8", kind="serve", slots=8, shortest=96, longest=640, count=32),
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["gemm", "gemm", "gemm", "gemv", "attention", "attention", "answer", "answer", "answer", "prompt", "serve", "serve"])
    if kind == "gemm":
        while True:
            col = rng.random() < 0.6
            m, n, k = _log(rng, 16, 8192), _log(rng, 64, 16384), 8 * _log(rng, 8, 1024)
            if not col:
                n = 8 * max(1, n // 8)
            if m * n * k <= 8192**3:
                return dict(kind=kind, m=m, n=n, k=k, b_col_maj=col, c_col_maj=rng.random() < 0.15)
    if kind == "gemv":
        return dict(kind=kind, m=_log(rng, 64, 128256), k=8 * _log(rng, 32, 1792))
    if kind == "attention":
        heads, kv_heads = rng.choice([(32, 8), (24, 8), (16, 4), (16, 16)])
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, d=rng.choice([64, 128]), seq=_log(rng, 48, 8192),
                    window=rng.choice([0, 0, 0, 1024]))
    if kind == "answer":
        model = rng.choice(["toy", "1b", "1b"])
        if model == "toy":
            turn = _log(rng, 1, 200)
            return dict(kind=kind, model=model, context=256, history=0, turn=turn, count=_log(rng, 2, 48), sampled=rng.random() < 0.3)
        context = rng.choice([2048, 8192, 16384])
        history = rng.choice([0, 0, _log(rng, 200, context * 3 // 4)])
        return dict(kind=kind, model=model, context=context, history=history, turn=_log(rng, 1, min(2000, context - history - 64)),
                    count=_log(rng, 4, 48), sampled=rng.random() < 0.3)
    if kind == "prompt":
        return dict(kind=kind, model="1b", context=8192, turn=_log(rng, 8, 7000))
    shortest = _log(rng, 8, 300)
    return dict(kind=kind, slots=rng.choice([1, 2, 4, 8]), shortest=shortest, longest=shortest + _log(rng, 1, 340), count=_log(rng, 4, 32))


# ---------------------------------------------------------------- inputs
def _device() -> torch.device:
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Normal:
    """Seeded bf16 tensors on the device."""

    def __init__(self, seed):
        self.g = torch.Generator(device=_device())
        self.g.manual_seed(int(seed))

    def __call__(self, *shape, scale=1.0, mean=0.0):
        return torch.randn(shape, generator=self.g, device=self.g.device).mul_(scale).add_(mean).to(BF16)

    def order(self, n):
        return torch.randperm(n, generator=self.g, device=self.g.device)


TOY = LlamaConfig(vocab_size=1024, hidden_size=512, num_hidden_layers=2, num_attention_heads=16, num_key_value_heads=4, head_dim=64,
                  intermediate_size=2048, rope_theta=500000.0, max_seq_len=256, prefill_chunk=256, eps=1e-5, tie_word_embeddings=False,
                  rope_scaling=Llama3RopeScaling(factor=8.0, low_freq_factor=1.0, high_freq_factor=4.0, original_max_position_embeddings=64))


def _llama(case, seed):
    """The config, the weights by checkpoint name, every token's successor, and the turns' tokens."""
    c = TOY if case["model"] == "toy" else dataclasses.replace(LLAMA_3_2_1B, tie_word_embeddings=False, prefill_chunk=2048)
    c = dataclasses.replace(c, max_seq_len=case["context"])
    normal, weights = _Normal(seed), {}
    for name, shape in llama_shapes(c).items():
        if len(shape) == 1:
            weights[name] = normal(*shape, scale=0.1, mean=1.0)
        elif "embed" in name:
            weights[name] = normal(*shape)
        else:
            joins = name.endswith(("o_proj.weight", "down_proj.weight"))
            weights[name] = normal(*shape, scale=0.02 * (2048 / c.hidden_size) ** 0.5 / (math.sqrt(2 * c.num_hidden_layers) if joins else 1))
    follows = _successors(weights, "model.embed_tokens.weight", "lm_head.weight", normal)
    tokens = np.random.default_rng(seed).integers(0, c.vocab_size, case.get("history", 0) + case["turn"])
    return c, weights, follows, tokens


def _successors(weights, embed, head, normal) -> np.ndarray:
    """Give the output matrix each token's embedding at its successor's row; the successors."""
    follows = normal.order(len(weights[embed]))
    weights[head] = torch.empty_like(weights[embed])
    weights[head][follows] = (weights[embed].float() * 0.02).to(BF16)
    return follows.cpu().numpy()


WIDTH, WINDOW = 2048, 1024


def _pufuzen(case, seed):
    """As ``_llama``, the tokens a list a request."""
    mlp = {"ff": 8192, "kind": "dense"}
    shared = {"heads": 16, "dim": 128, "vdim": 128, "q_rank": 1536, "kv_rank": 512}
    recurrent = {"type": "mingru", "mixer": {"width": WIDTH}, "mlp": None}
    windowed = {"type": "latent_attention", "mlp": mlp, "mixer": {**shared, "scale": 128**-0.5, "mask": {"size": WINDOW}}}
    causal = {"type": "latent_attention_2", "mlp": mlp, "mixer": {**shared, "rot_dim": 64, "rot": {"base": 10000.0, "dims": 64},
                                                                   "scale": 192**-0.5}}
    c = PufuzenConfig(vocab_size=128256, hidden_size=WIDTH, layers=tuple([recurrent, recurrent, windowed, causal] * 4), eps=1e-5,
                      max_seq_len=4096, prefill_chunk=2048, slots=case["slots"])
    normal, weights = _Normal(seed), {}
    for name, shape in pufuzen_shapes(c).items():
        leaf = name.split(".", 1)[-1]
        if "norm" in leaf:
            weights[name] = normal(*shape, scale=0.1, mean=1.0)
        elif leaf == "mlp.act":
            weights[name] = torch.tensor([0.7, 0.5, -0.4, 0.2], device=_device()).to(BF16)
        elif leaf == "mix.z.b":
            weights[name] = normal(*shape, scale=1.5, mean=-2.0)
        elif len(shape) == 1:
            weights[name] = normal(*shape, scale=0.3)
        elif leaf == "embed":
            weights[name] = normal(*shape)
        elif leaf != "head":
            weights[name] = normal(*shape, scale=0.02 / (math.sqrt(24) if leaf in ("mix.o", "mlp.down") else 1))
    follows = _successors(weights, "embed", "head", normal)
    rng = np.random.default_rng(seed)
    lengths = rng.integers(case["shortest"], case["longest"] + 1, case["slots"])
    return c, weights, follows, [rng.integers(0, c.vocab_size, n).tolist() for n in lengths]


def prepare(case, seed):
    kind, s = case["kind"], SimpleNamespace(case=case)
    if kind == "gemm":
        s.a, s.b = _matrices(case, seed)
        s.c = torch.empty((case["n"], case["m"]) if case["c_col_maj"] else (case["m"], case["n"]), dtype=BF16, device=s.a.device)
    elif kind == "gemv":
        normal = _Normal(seed)
        s.w, s.x = normal(case["m"], case["k"], scale=0.02), normal(case["k"])
        s.y = torch.empty(case["m"], dtype=BF16, device=s.x.device)
    elif kind == "attention":
        s.q, s.k, s.v = _heads(case, seed)
        s.o = torch.empty_like(s.q)
    elif kind == "serve":
        c, weights, _, s.prompts = _pufuzen(case, seed)
        s.model = Pufuzen(c, weights)
        s.model.load_versions()
    else:
        c, weights, _, tokens = _llama(case, seed)
        s.model = Llama(c, weights)
        s.model.load_versions()
        s.tokens, s.held = tokens.tolist(), case.get("history", 0)
        if s.held:
            s.model.logits(s.tokens[: s.held])
    return s


def _matrices(case, seed):
    normal = _Normal(seed)
    m, n, k = case["m"], case["n"], case["k"]
    return normal(m, k), normal(*((n, k) if case["b_col_maj"] else (k, n)), scale=0.02)


def _heads(case, seed):
    """Queries and keys of unit variance, as a layer's projections of normed rows give them; row by row."""
    normal, d, seq = _Normal(seed), case["d"], case["seq"]
    return normal(seq, case["heads"], d), normal(seq, case["kv_heads"], d), normal(seq, case["kv_heads"], d)


# ---------------------------------------------------------------- one pass
def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "gemm":
        K.gemm(s.a, s.b, s.c, M=case["m"], N=case["n"], K=case["k"], b_col_maj=case["b_col_maj"], c_col_maj=case["c_col_maj"])
        return s.c
    if kind == "gemv":
        K.gemv(s.w, s.x, s.y, M=case["m"], K=case["k"])
        return s.y
    if kind == "attention":
        K.mha_prefill(s.q, s.k, s.v, s.o, heads=case["heads"], kv_heads=case["kv_heads"], d=case["d"], seq=case["seq"], kv_len=case["seq"],
                      window=case["window"] - 1 if case["window"] else None, q_interleaved=True, kv_interleaved=True)
        return s.o
    if kind == "serve":
        # The requests are answered as one batch, and the answers scored: the logits behind each.
        answers = s.model.generate_batch(s.prompts, case["count"])
        entries = [Entry(i, p + a, [len(p) + len(a) - 1]) for i, (p, a) in enumerate(zip(s.prompts, answers))]
        scores = s.model.batch.step(entries)
        for e in entries:
            s.model.batch.end(e.key)
        return {"tokens": np.asarray(answers), "logits": np.concatenate(scores)}
    s.model.session.forget(s.held)   # the turn is asked anew
    if kind == "prompt":
        return s.model.logits(s.tokens)
    sampler = Sampler(temperature=0.7, top_k=50) if case["sampled"] else None
    answer = s.model.generate(s.tokens, case["count"], sampler)
    return {"tokens": np.asarray(answer), "logits": s.model.logits(s.tokens + answer)}


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind == "gemv":
        m, k = case["m"], case["k"]
        return {"bytes": 2 * (m * k + m + k), "flops": 2 * m * k}
    if kind == "attention":
        s, w = case["seq"], case["window"] or case["seq"]
        pairs = sum(min(i + 1, w) for i in range(s))
        return {"bytes": 4 * s * case["d"] * (case["heads"] + case["kv_heads"]), "flops": 4 * case["heads"] * case["d"] * pairs}
    if kind == "serve":
        # Every matrix of a layer once a token; weights read once by the prompts, once by each step and once by the scoring.
        recurrent = 5 * WIDTH * WIDTH
        feed = 2 * 8192 * WIDTH + WIDTH * WIDTH
        latent = WIDTH * (1536 + 512 + WIDTH) + 1536 * 16 * 128 + 512 * 16 * 256 + WIDTH * WIDTH + feed
        layers = 4 * (2 * recurrent + 2 * latent + WIDTH * 64 + 1536 * 16 * 64)
        head, mean, count, slots = 128256 * WIDTH, (case["shortest"] + case["longest"]) / 2, case["count"], case["slots"]
        return {"bytes": 2 * (layers + head) * (count + 1), "flops": 2 * slots * (layers * (2 * mean + 2 * count) + head * (count + 1))}
    c = TOY if case["model"] == "toy" else LLAMA_3_2_1B
    e, h, g, d, f = c.hidden_size, c.num_attention_heads, c.num_key_value_heads, c.head_dim, c.intermediate_size
    layer, head = e * d * (2 * h + 2 * g) + 3 * e * f, e * c.vocab_size
    held, turn, count = case.get("history", 0), case["turn"], case.get("count", 0)
    passes = 1 + count                       # the prompt, the steps of the draws behind the first, the scored token
    keys = sum(held + turn + i for i in range(count + 1))
    pairs = sum(held + i + 1 for i in range(turn)) + keys
    return {"bytes": 2 * passes * (c.num_hidden_layers * layer + head) + 4 * c.num_hidden_layers * g * d * keys,
            "flops": 2 * (c.num_hidden_layers * layer * (turn + count) + head * passes) + 4 * c.num_hidden_layers * h * d * pairs}


def tolerance(case):
    """About four times what two orders of the same sums differ by: a bf16 result's last bit, and in a decoder what its layers make
    of such bits in the rows they pass on."""
    return TOLERANCES[case["kind"]]


TOLERANCES = {"gemm": {"rel": 2e-3, "max": 0.01}, "gemv": {"rel": 2e-3, "max": 0.01}, "attention": {"rel": 6e-3, "max": 0.1},
              "answer": {"rel": 0.02, "max": 0.15, "differ": 0.0}, "prompt": {"rel": 0.02, "max": 0.15},
              "serve": {"rel": 0.008, "max": 0.05, "differ": 0.0}}


# ---------------------------------------------------------------- the same in 64 bits
def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        a, b = (t.double() for t in _matrices(case, seed))
        c = a @ (b.t() if case["b_col_maj"] else b)
        return c.t().contiguous() if case["c_col_maj"] else c
    if kind == "gemv":
        normal = _Normal(seed)
        w, x = normal(case["m"], case["k"], scale=0.02).double(), normal(case["k"]).double()
        return w @ x
    if kind == "attention":
        q, k, v = (t.double() for t in _heads(case, seed))
        return _attend(q, k, v, case["d"] ** -0.5, window=case["window"])
    if kind == "serve":
        c, weights, follows, prompts = _pufuzen(case, seed)
        answers = [_chain(follows, p[-1], case["count"]) for p in prompts]
        logits = [_pufuzen_logits(c, weights, p + a, case["count"]) for p, a in zip(prompts, answers)]
        for rows, a in zip(logits, answers):
            _check(rows, a)
        return {"tokens": np.asarray(answers), "logits": torch.stack([rows[-1] for rows in logits])}
    c, weights, follows, tokens = _llama(case, seed)
    tokens, count = tokens.tolist(), case.get("count", 0)
    answer = _chain(follows, tokens[-1], count)
    rows = _llama_logits(c, weights, tokens + answer, count)
    if kind == "prompt":
        return rows[-1]
    _check(rows, answer)
    return {"tokens": np.asarray(answer), "logits": rows[-1]}


def _chain(follows, token, count) -> list[int]:
    out = []
    for _ in range(count):
        token = int(follows[token])
        out.append(token)
    return out


def _check(rows, answer) -> None:
    """The tokens are the best ones of the logits before each."""
    if rows[:-1].argmax(-1).tolist() != answer:
        raise AssertionError("a successor is not the most likely token")


def _normed(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w


def _attend(q, k, v, scale, window=0, sink=None):
    """q (T, H, D), k (T, G, D), v (T, G, V): causal, a block of queries at a time."""
    T, H, _ = q.shape
    group, out = H // k.shape[1], torch.empty(T, H, v.shape[-1], dtype=q.dtype, device=q.device)
    for first in range(0, T, 1024):
        last = min(T, first + 1024)
        low = max(0, first - window + 1) if window else 0
        i, j = torch.arange(first, last, device=q.device)[:, None], torch.arange(low, last, device=q.device)[None]
        hidden = (j > i) | (j <= i - window) if window else j > i
        for h in range(H):
            s = q[first:last, h] @ k[low:last, h // group].t() * scale
            s.masked_fill_(hidden, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[h].expand(last - first, 1)], dim=1)
            out[first:last, h] = torch.softmax(s, -1)[:, : last - low] @ v[low:last, h // group]
    return out


def _llama_logits(c, weights, tokens, count):
    """The logits behind the last ``count + 1`` tokens."""
    w = {n: t for n, t in weights.items()}
    e, h, g, d = c.hidden_size, c.num_attention_heads, c.num_key_value_heads, c.head_dim
    x = w["model.embed_tokens.weight"][torch.as_tensor(tokens, device=_device())].double()
    f = c.rope_theta ** (-torch.arange(0, d, 2, device=x.device).double() / d)
    r = c.rope_scaling
    wavelength = 2 * math.pi / f
    share = (r.original_max_position_embeddings / wavelength - r.low_freq_factor) / (r.high_freq_factor - r.low_freq_factor)
    share = share.clamp(0, 1)
    f = (1 - share) * f / r.factor + share * f
    angle = torch.arange(len(tokens), device=x.device).double()[:, None, None] * f
    cos, sin = angle.cos(), angle.sin()

    def turned(y):
        a, b = y[..., : d // 2], y[..., d // 2 :]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    for i in range(c.num_hidden_layers):
        name = f"model.layers.{i}."

        def matrix(n, name=name):
            return w[name + n + ".weight"].double()

        y = _normed(x, matrix("input_layernorm"), c.eps)
        q, k, v = ((y @ matrix(f"self_attn.{n}_proj").t()).reshape(len(tokens), -1, d) for n in "qkv")
        a = _attend(turned(q), turned(k), v, d**-0.5)
        x = x + a.reshape(len(tokens), h * d) @ matrix("self_attn.o_proj").t()
        y = _normed(x, matrix("post_attention_layernorm"), c.eps)
        y = torch.nn.functional.silu(y @ matrix("mlp.gate_proj").t()) * (y @ matrix("mlp.up_proj").t())
        x = x + y @ matrix("mlp.down_proj").t()
    x = _normed(x[-count - 1 :], w["model.norm.weight"].double(), c.eps)
    return x @ w["lm_head.weight"].double().t()


def _pufuzen_logits(c, weights, tokens, count):
    """As ``_llama_logits``."""
    w = {n: t.double() for n, t in weights.items() if n not in ("embed", "head")}
    T = len(tokens)
    x = weights["embed"][torch.as_tensor(tokens, device=_device())].double()
    for i, spec in enumerate(c.layers):
        name, m = f"l{i}.", spec["mixer"]
        mix = name + "mix."
        y = _normed(x, w[name + "norm1"], c.eps)
        if spec["type"] == "mingru":
            z, u = torch.sigmoid(y @ w[mix + "z"].t() + w[mix + "z.b"]), y @ w[mix + "x"].t() + w[mix + "x.b"]
            moved, kept = z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u)), 1 - z
            states = torch.empty_like(moved)
            state = torch.zeros_like(moved[0])
            for t in range(T):
                state = torch.addcmul(moved[t], kept[t], state)
                states[t] = state
            out = (states * torch.nn.functional.silu(y @ w[mix + "g"].t())) @ w[mix + "o"].t()
        else:
            H, D, R, rot = m["heads"], m["dim"], m["kv_rank"], m.get("rot_dim", 0)
            q = (_normed(y @ w[mix + "dq"].t(), w[mix + "dq.norm"], c.eps) @ w[mix + "uq"].t()).reshape(T, H, D + rot)
            down = y @ w[mix + "dkv"].t()
            latent = _normed(down[:, :R], w[mix + "dkv.norm"], c.eps)
            k, v = (latent @ w[mix + "uk"].t()).reshape(T, H, D), (latent @ w[mix + "uv"].t()).reshape(T, H, -1)
            if rot:
                f = m["rot"]["base"] ** (-torch.arange(0, rot, 2, device=x.device).double() / rot)
                angle = torch.arange(T, device=x.device).double()[:, None, None] * f
                q = torch.cat([q[..., :D], _pairs_turned(q[..., D:], angle)], -1)
                k = torch.cat([k, _pairs_turned(down[:, None, R:], angle).expand(T, H, rot)], -1)
            out = _attend(q, k, v, m["scale"], window=m["mask"]["size"] if "mask" in m else 0, sink=w.get(mix + "sink"))
            out = out.reshape(T, -1) @ w[mix + "o"].t()
        x = x + torch.sigmoid(y @ w[name + "rg1"].t() + w[name + "rg1.b"]) * out
        if spec["mlp"] is not None:
            y = _normed(x, w[name + "norm2"], c.eps)
            z = y @ w[name + "mlp.up"].t() + w[name + "mlp.up.b"]
            act = w[name + "mlp.act"]
            z = sum(act[p - 1] * _normed(z**p, 1.0, c.eps) for p in (1, 2, 3)) + act[3]
            out = z @ w[name + "mlp.down"].t() + w[name + "mlp.down.b"]
            x = x + torch.sigmoid(y @ w[name + "rg2"].t() + w[name + "rg2.b"]) * out
    x = _normed(x[-count - 1 :], w["final.norm"], c.eps)
    return x @ weights["head"].double().t() * c.logit_scale


def _pairs_turned(y, angle):
    a, b = y[..., 0::2], y[..., 1::2]
    return torch.stack([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1).flatten(-2)
