"""Cases by which the speed of the framework's text path is measured.

Text generation is what the framework is for in the first place: a prompt goes in, logits or tokens
come out.  A program reaches it in three ways, and each is a kind of case here:

* ``prompt``: ``model.prefill_logits``, the logits after a whole prompt (time to first token,
  scoring);
* ``request``: ``DeviceDecoder.start`` and ``run_decode``, a prompt and the tokens after it, one
  replay of the captured step per token (a chat reply);
* ``serve``: ``model.step``, several sequences side by side, their prompts in one ragged step and
  then one token of each per step (a server, a trace).  The hybrid designs only: a Llama model
  holds one sequence at a time and its server queues requests.

Models are the three families at the sizes of the repository's own design bench (nine layer runs of
the width, heads and feed-forward of 1B, 8B and 70B decoders), with random weights, in the two
16-bit types that the decode kernels take.  32-bit models run the vendor's product and are there for
checks; images have a benchmark of their own.

Greedy tokens of random weights hang on ties.  A trained model is sure of most of its tokens, so the
heads here prefer one follower of each token (the tied head of Navalorn prefers the token itself) by
a wide margin, and the embedding of a token of a design with experts holds the router directions of
the experts that suit it, a random set for each token, as trained routers are even and sure.
"""
from __future__ import annotations

import math

import torch

from cake_amd.models.base import StepEntry
from cake_amd.models.decoder import DeviceDecoder
from cake_amd.models.hybrid.bench import DESIGNS, SIZES, llama_config
from cake_amd.models.hybrid.model import HybridModel
from cake_amd.models.hybrid.weights import random_tensors, tensor_shapes
from cake_amd.models.llama3.blocks import LayerStack
from cake_amd.models.llama3.decode_loop import run_decode
from cake_amd.models.llama3.model import LlamaModel
from cake_amd.models.llama3.weights import BLOCK_TENSORS, BlockWeights, HeadWeights, layer_name

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
FOLLOW = 17                     # the token that a head prefers after t is t + FOLLOW
PENALTY, LAST_N = 1.1, 128      # the generator's defaults
PLANT = 60.0                    # router directions in an embedding row
SURE = 0.7                      # scale of the linear weights where routers read the rows


def listed() -> list[dict]:
    def case(name, family, size, kind, dtype, **kw):
        return dict(name=name, family=family, size=size, kind=kind, dtype=dtype, **kw)
    return [
        # the smallest call: a command or a few words, latency and launches
        case("llama 1B prompt 5", "llama", "w2048", "prompt", "bf16", tokens=5),
        # a short question without history
        case("llama 8B prompt 45", "llama", "w4096", "prompt", "bf16", tokens=45),
        # a question with some history or a retrieved paragraph
        case("llama 8B prompt 777", "llama", "w4096", "prompt", "f16", tokens=777),
        # a document
        case("llama 8B prompt 6000", "llama", "w4096", "prompt", "bf16", tokens=6000),
        # a chat reply
        case("llama 8B chat", "llama", "w4096", "request", "bf16", tokens=33, new=40),
        # a reply late in a long conversation, at the width of the largest model
        case("llama 70B reply", "llama", "w8192", "request", "f16", tokens=1490, new=24),
        # the hybrid designs: a document, a reply, a server's batch
        case("fonapel 8B prompt 1100", "fonapel", "w4096", "prompt", "bf16", tokens=1100),
        case("fonapel 1B chat", "fonapel", "w2048", "request", "f16", tokens=210, new=40),
        case("fonapel 8B serve 24", "fonapel", "w4096", "serve", "bf16", seqs=24, tokens=60, new=6),
        case("navalorn 8B prompt 2048", "navalorn", "w4096", "prompt", "bf16", tokens=2048),
        case("navalorn 8B chat", "navalorn", "w4096", "request", "bf16", tokens=90, new=24),
        case("navalorn 1B serve 13", "navalorn", "w2048", "serve", "f16", seqs=13, tokens=90, new=6),
    ]


def _log(rng, lo: int, hi: int) -> int:
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng) -> dict:
    """One more case: families, sizes, kinds and types evenly; lengths over their logarithm."""
    most = max(_cost(c) for c in listed())
    while True:
        family = rng.choice(("llama", "fonapel", "navalorn"))
        kind = rng.choice(("prompt", "request") if family == "llama" else
                          ("prompt", "request", "serve"))
        c = dict(family=family, kind=kind, dtype=rng.choice(("bf16", "f16")),
                 size=rng.choice(("w2048", "w4096", "w8192") if family == "llama" else
                                 ("w2048", "w4096")))
        if kind == "prompt":
            c["tokens"] = _log(rng, 2, 6000)
        elif kind == "request":
            c.update(tokens=_log(rng, 8, 2000), new=_log(rng, 8, 48))
        else:
            c.update(seqs=_log(rng, 2, 32), tokens=_log(rng, 8, 200), new=_log(rng, 2, 8))
        if _cost(c) <= most:
            return c


# ---------------------------------------------------------------------------- inputs
def _config(case):
    if case["family"] == "llama":
        return llama_config(case["size"])
    return DESIGNS[case["family"]](case["size"])


def _llama_tensors(cfg, dtype, seed: int):
    """A getter of a checkpoint's tensors: linear weights that keep the size of what they read, a
    head that prefers the token FOLLOW after the last one."""
    H, I, V = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size
    nq, nk = cfg.num_attention_heads * cfg.head_dim, cfg.num_key_value_heads * cfg.head_dim
    shapes = {"wq": (nq, H), "wk": (nk, H), "wv": (nk, H), "wo": (H, nq), "wg": (I, H),
              "wu": (I, H), "wd": (H, I)}
    key = {suffix: k for k, suffix in BLOCK_TENSORS}

    def get(name: str) -> torch.Tensor:
        g = torch.Generator(device=DEV)
        g.manual_seed(seed * 1000003 + sum((i + 1) * ord(ch) for i, ch in enumerate(name)))
        if name == "lm_head.weight":
            return torch.roll(get("model.embed_tokens.weight"), FOLLOW, 0) * H ** -0.5
        if name == "model.embed_tokens.weight":
            return torch.empty((V, H), device=DEV, dtype=dtype).normal_(0.0, 1.0, generator=g)
        shape = shapes.get(key.get(name.split(".", 3)[-1], ""))
        if shape is None:   # a norm
            return torch.empty(H, device=DEV, dtype=dtype).normal_(1.0, 0.05, generator=g)
        return torch.empty(shape, device=DEV, dtype=dtype).normal_(0.0, shape[1] ** -0.5, generator=g)
    return get


def _hybrid_tensors(cfg, dtype, seed: int):
    """The repository's random tensors, with a sure head and sure routers."""
    W = cfg.hidden_size
    moe = [L.mlp for L in cfg.layers if L.mlp is not None and L.mlp.kind == "experts"]
    experts, top = (moe[0].experts, moe[0].top) if moe else (0, 0)
    raw = random_tensors(cfg, DEV, dtype, seed, gain=SURE if moe else 1.0)

    def directions():
        g = torch.Generator(device=DEV).manual_seed(seed * 7919 + 5)
        r = torch.randn(experts, W, device=DEV, generator=g)
        return r / r.norm(dim=1, keepdim=True)

    def get(name: str) -> torch.Tensor:
        if name == "head":
            return torch.roll(get("embed"), FOLLOW, 0) * W ** -0.5
        if name == "loop.in":     # a pass continues the row that it is entered with
            t = raw(name)
            t[:, :W] += torch.eye(W, device=DEV, dtype=t.dtype)
            return t
        if experts and name.endswith(".router"):
            return directions().to(dtype)
        if experts and name == "embed":
            t = raw(name).float()
            g = torch.Generator(device=DEV).manual_seed(seed * 7919 + 6)
            best = torch.rand(t.shape[0], experts, device=DEV, generator=g).topk(top, 1).indices
            pick = torch.zeros(t.shape[0], experts, device=DEV).scatter_(1, best, PLANT)
            t += pick @ directions()
            return (t * (W / t.pow(2).sum(1, keepdim=True)).sqrt()).to(dtype)
        return raw(name)
    return get


def _tensors(case, seed: int):
    cfg, dtype = _config(case), DTYPES[case["dtype"]]
    return cfg, (_llama_tensors if case["family"] == "llama" else _hybrid_tensors)(cfg, dtype, seed)


def _ids(cfg, n: int, seed: int) -> list[int]:
    return torch.randint(0, cfg.vocab_size, (n,),
                         generator=torch.Generator().manual_seed(seed)).tolist()


def _lengths(case) -> list[int]:
    """Prompt lengths of a serve case: from a quarter of `tokens` to almost twice of it, ragged."""
    return [max(1, case["tokens"] * (1 + (5 * i + 3) % 7) // 4) for i in range(case["seqs"])]


def _sequences(case, cfg, seed: int) -> list[list[int]]:
    """Of a serve case: each sequence's prompt and the tokens fed after it."""
    return [_ids(cfg, n + case["new"], seed * 4096 + i) for i, n in enumerate(_lengths(case))]


def _model(case, cfg, get, max_seq: int):
    dtype = DTYPES[case["dtype"]]
    if case["family"] == "llama":
        w = {i: BlockWeights.load(get, layer_name(i), cfg, DEV, dtype)
             for i in range(cfg.num_hidden_layers)}
        stack = LayerStack(cfg, w, DEV, dtype, max_seq, "hip")
        return LlamaModel(cfg, HeadWeights.load(get, cfg, DEV, dtype), stack)
    return HybridModel.build(cfg, get, DEV, dtype, max_seq, slots=case.get("seqs", 1) + 1)


def prepare(case: dict, seed: int) -> dict:
    cfg, get = _tensors(case, seed)
    if case["kind"] == "serve":
        most = max(_lengths(case)) + case["new"] + 1
    else:
        most = case["tokens"] + case.get("new", 0) + 2
    model = _model(case, cfg, get, -(-most // 64) * 64)
    state = {"kind": case["kind"], "model": model, "new": case.get("new", 0)}
    if case["kind"] == "serve":
        state["seqs"] = _sequences(case, cfg, seed)
        return state
    state["prompt"] = _ids(cfg, case["tokens"], seed)
    if case["kind"] == "prompt":
        state["logits"] = torch.empty(cfg.vocab_size, device=DEV, dtype=torch.float32)
    else:
        dec = state["dec"] = DeviceDecoder(model, repeat_penalty=PENALTY, repeat_last_n=LAST_N)
        dec.start(state["prompt"])
        dec.capture()
    return state


@torch.no_grad()
def run(state: dict):
    model = state["model"]
    if state["kind"] == "prompt":
        model.prefill_logits(state["prompt"], state["logits"])
        return state["logits"]
    if state["kind"] == "request":
        dec = state["dec"]
        first = dec.start(state["prompt"])
        rest = run_decode(dec, state["new"]).tokens
        return {"tokens": torch.tensor([first, *rest]), "logits": dec.logits()}
    new = state["new"]
    seqs = [(model.open_sequence(), s) for s in state["seqs"]]
    out = [model.step([StepEntry(i, s[:len(s) - new], [len(s) - new - 1]) for i, s in seqs])]
    for k in range(new):
        out.append(model.step([StepEntry(i, [s[len(s) - new + k]], [0]) for i, s in seqs]))
    for i, _ in seqs:
        model.close_sequence(i)
    return [torch.cat(x) for x in out]


# ---------------------------------------------------------------------------- work, tolerance
def _steps(case) -> list[list[tuple[int, int]]]:
    """Per step: (tokens fed, tokens held before) of every sequence."""
    if case["kind"] == "serve":
        n = _lengths(case)
        return [[(x, 0) for x in n]] + [[(1, x + k) for x in n] for k in range(case["new"])]
    return [[(case["tokens"], 0)]] + [[(1, case["tokens"] + k)] for k in range(case.get("new", 0))]


def _layers(cfg):
    """Per layer run: (weights that every token uses, of one expert, experts, used per token,
    multiply-adds per query and key, cached values per position, recurrent 32-bit values)."""
    if not hasattr(cfg, "layers"):
        hd = cfg.head_dim
        return [(cfg.layer_bytes(1), 0, 0, 0, 2 * cfg.num_attention_heads * hd,
                 2 * cfg.num_key_value_heads * hd, 0)] * cfg.num_hidden_layers
    sizes: dict[int, int] = {}
    for n, s in tensor_shapes(cfg).items():
        if n[0] == "l" and n[1].isdigit() and ".mlp.e" not in n:
            i = int(n[1:n.index(".")])
            sizes[i] = sizes.get(i, 0) + math.prod(s)
    out = []
    for r in cfg.runs():
        m, f = cfg.layers[r.layer].mixer, cfg.layers[r.layer].mlp
        dense = sizes[cfg.weights_layer(r.layer)]
        if r.enter is not None:
            dense += 2 * cfg.hidden_size ** 2
        one, n, top = (2 * cfg.hidden_size * f.ff, f.experts, f.top) \
            if f is not None and f.kind == "experts" else (0, 0, 0)
        if m.kind == "latent":
            att, held, rec = m.heads * (m.dim + m.rot_dim + m.vdim), m.kv_rank + m.rot_dim, 0
        elif m.kind == "attention":
            att, held, rec = m.heads * (m.dim + m.vdim), m.kv_heads * (m.dim + m.vdim), 0
        else:   # the state's update and its read-out, per token
            att, held, rec = 0, 0, m.heads * m.dim * m.vdim
        out.append((dense, one, n, top, att, held, rec))
    return out


def work(case: dict) -> dict:
    cfg = _config(case)
    V, H = cfg.vocab_size, cfg.hidden_size
    flops = size = 0.0
    layers = _layers(cfg)
    for step in _steps(case):
        n, B = sum(t for t, _ in step), len(step)
        pairs = sum(t * p + t * (t + 1) // 2 for t, p in step)
        for dense, one, experts, top, att, held, rec in layers:
            flops += 2.0 * n * (dense + top * one) + 2.0 * pairs * att + 6.0 * n * rec
            size += 2.0 * (dense + min(experts, n * top) * one)
            size += 2.0 * held * sum(2 * t + p for t, p in step if held) - 2.0 * held * n
            size += 4.0 * rec * sum(2 if p else 1 for _, p in step)
        flops += 2.0 * B * V * H
        size += 2.0 * V * H + 4.0 * B * V + 2.0 * n * H
    return {"bytes": size, "flops": flops}


def _cost(case) -> float:
    """Seconds, roughly: at half the card's rates and some time per step."""
    w = work(case)
    return w["flops"] / 1.2e15 + w["bytes"] / 4e12 + 1e-4 * len(_steps(case))


def tolerance(case: dict) -> dict:
    """Of the logits: four times the largest error of the listed cases against 64 bits (0.006 in
    bf16, 0.0009 in f16), which is the rounding of the activations between the projections."""
    return {"rel": 0.024 if case["dtype"] == "bf16" else 0.0036, "max": 0.2, "differ": 0.0}


# ---------------------------------------------------------------------------- 64 bits
D = torch.float64


def _rms(x, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _lnorm(x, w, eps):
    x = x - x.mean(-1, keepdim=True)
    return _rms(x, eps) * w


def _causal(q, k, v, scale, sink=False):
    """q, k [T, heads, d], v [T, heads, e] -> [T, heads, e]."""
    T, H = q.shape[:2]
    out = torch.empty(T, H, v.shape[2], dtype=D, device=q.device)
    hidden = torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1)
    for h in range(H):
        s = (q[:, h] @ k[:, h].t() * scale).masked_fill_(hidden, -math.inf)
        top = s.amax(-1, keepdim=True).clamp_(min=0.0 if sink else -math.inf)
        s = (s - top).exp_()
        out[:, h] = (s @ v[:, h]) / (s.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0.0))
    return out


def _turn_halves(x, theta):
    T, _, d = x.shape
    f = theta ** (-torch.arange(0, d, 2, dtype=D, device=x.device) / d)
    a = (torch.arange(T, dtype=D, device=x.device)[:, None] * f)[:, None]
    u, v = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([u * a.cos() - v * a.sin(), u * a.sin() + v * a.cos()], -1)


def _turn_pairs(x, rot):
    n = rot.dims // 2
    f = torch.tensor(_frequencies(rot), dtype=D, device=x.device)
    mag = 1.0 if rot.scaling is None else 0.1 * math.log(rot.scaling.factor) + 1.0
    a = (torch.arange(x.shape[0], dtype=D, device=x.device)[:, None] * f)[:, None]
    u, v = x[..., 0:2 * n:2], x[..., 1:2 * n:2]
    y = x.clone()
    y[..., 0:2 * n:2] = (u * a.cos() - v * a.sin()) * mag
    y[..., 1:2 * n:2] = (v * a.cos() + u * a.sin()) * mag
    return y


def _frequencies(rot):
    f, s = [rot.base ** (-2.0 * i / rot.dims) for i in range(rot.dims // 2)], rot.scaling
    if s is None:
        return f

    def dim_of(turns):
        return rot.dims * math.log(s.original / (2 * math.pi * turns)) / (2 * math.log(rot.base))
    lo = max(math.floor(dim_of(s.fast)), 0)
    hi = min(math.ceil(dim_of(s.slow)), rot.dims - 1)
    ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(len(f))]
    return [x / s.factor * r + x * (1 - r) for x, r in zip(f, ramp)]


def _llama_rows(cfg, w, ids):
    nh, nk, hd, eps = (cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim,
                       cfg.rms_norm_eps)
    x = w("model.embed_tokens.weight")[ids]
    T = x.shape[0]
    for i in range(cfg.num_hidden_layers):
        t = {k: f"model.layers.{i}.{s}" for k, s in BLOCK_TENSORS}
        h = _rms(x, eps) * w(t["ln1"])
        q = _turn_halves((h @ w(t["wq"]).t()).view(T, nh, hd), cfg.rope_theta)
        k = _turn_halves((h @ w(t["wk"]).t()).view(T, nk, hd), cfg.rope_theta)
        v = (h @ w(t["wv"]).t()).view(T, nk, hd)
        k, v = (z.repeat_interleave(nh // nk, 1) for z in (k, v))
        x = x + _causal(q, k, v, hd ** -0.5).reshape(T, -1) @ w(t["wo"]).t()
        h = _rms(x, eps) * w(t["ln2"])
        g = h @ w(t["wg"]).t()
        x = x + (g * torch.sigmoid(g) * (h @ w(t["wu"]).t())) @ w(t["wd"]).t()
    return _rms(x, eps) * w("model.norm.weight"), w("lm_head.weight")


def _delta(h, w, p, m, eps):
    T, H, G = h.shape[0], m.heads, m.kv_heads

    def conv(name):
        x, c = h @ w(p + name).t(), w(p + name + ".conv")
        z = torch.cat([x.new_zeros(m.taps - 1, x.shape[1]), x])
        y = sum(z[j:j + T] * c[:, j] for j in range(m.taps))
        return y * torch.sigmoid(y)
    q, k, v = conv("q").view(T, G, m.dim), conv("k").view(T, G, m.dim), conv("v").view(T, H, m.vdim)
    q = q * torch.rsqrt(q.pow(2).sum(-1, keepdim=True) + 1e-6) * m.dim ** -0.5
    k = k * torch.rsqrt(k.pow(2).sum(-1, keepdim=True) + 1e-6)
    q, k = (z.repeat_interleave(H // G, 1) for z in (q, k))
    beta = torch.sigmoid(h @ w(p + "b").t())
    decay = torch.exp(-w(p + "A_log").exp() *
                      torch.nn.functional.softplus(h @ w(p + "a").t() + w(p + "dt_bias"),
                                                   threshold=40.0))
    S = h.new_zeros(H, m.dim, m.vdim)
    o = h.new_empty(T, H, m.vdim)
    for t in range(T):
        S = S * decay[t][:, None, None]
        u = beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None], S)[:, 0])
        S = S + k[t][:, :, None] * u[:, None]
        o[t] = torch.bmm(q[t][:, None], S)[:, 0]
    z = (h @ w(p + "g").t()).view(T, H, m.vdim)
    return (_rms(o, eps) * w(p + "norm") * z * torch.sigmoid(z)).reshape(T, -1) @ w(p + "o").t()


def _attention(h, w, p, m, eps):
    T, H, G = h.shape[0], m.heads, m.kv_heads
    q = _rms(_turn_pairs((h @ w(p + "q").t()).view(T, H, m.dim), m.rot), eps)
    k = _rms(_turn_pairs((h @ w(p + "k").t()).view(T, G, m.dim), m.rot), eps)
    v = (h @ w(p + "v").t()).view(T, G, m.vdim)
    k, v = (z.repeat_interleave(H // G, 1) for z in (k, v))
    o = _causal(q, k, v, m.scale, sink=True).reshape(T, -1)
    return (o * torch.sigmoid(h @ w(p + "g").t())) @ w(p + "o").t()


def _latent(h, w, p, m, eps):
    T, H = h.shape[0], m.heads
    c = _rms(h @ w(p + "dq").t(), eps) * w(p + "dq.norm")
    q = (c @ w(p + "uq").t()).view(T, H, m.dim + m.rot_dim)
    q = torch.cat([q[..., :m.dim], _turn_pairs(q[..., m.dim:], m.rot)], -1)
    d = h @ w(p + "dkv").t()
    c = _rms(d[:, :m.kv_rank], eps) * w(p + "dkv.norm")
    r = _turn_pairs(d[:, None, m.kv_rank:], m.rot).expand(T, H, m.rot_dim)
    k = torch.cat([(c @ w(p + "uk").t()).view(T, H, m.dim), r], -1)
    v = (c @ w(p + "uv").t()).view(T, H, m.vdim)
    return _causal(q, k, v, m.scale).reshape(T, -1) @ w(p + "o").t()


def _routed(h, w, p, f):
    s, e = torch.sigmoid(h @ w(p + "router").t()).topk(f.top, -1)
    out = torch.zeros_like(h)
    for i in range(f.experts):
        t, j = (e == i).nonzero(as_tuple=True)
        if t.numel():
            a = ((h[t] * s[t, j, None]) @ w(f"{p}e{i}.up").t()).clamp_(min=0.0).pow(2)
            out.index_add_(0, t, a @ w(f"{p}e{i}.down").t())
    return out


def _hybrid_rows(cfg, w, ids):
    eps, W = cfg.eps, cfg.hidden_size
    x = w("embed")[ids]
    if cfg.embed_norm:
        x = _lnorm(x, w("embed.norm"), eps)
    x0 = x

    def norm(x, name):
        return _lnorm(x, w(name), eps) if cfg.layer_norm else _rms(x, eps) * (1 + w(name))
    for r in cfg.runs():
        i = cfg.weights_layer(r.layer)
        L, p = cfg.layers[i], f"l{i}.mlp."
        m, f = L.mixer, L.mlp
        if r.enter is not None:
            x = torch.cat([x, x0], -1) @ w("loop.in").t() + w("loop.step")[r.enter]
        h = norm(x, f"l{i}.norm1")
        y = {"attention": _attention, "delta": _delta, "latent": _latent}[m.kind](
            h, w, f"l{i}.mix.", m, eps)
        if L.parallel:
            u = h @ w(p + "up").t()
            y = y + (0.5 * u * (1 + torch.erf(u / math.sqrt(2.0)))) @ w(p + "down").t()
            x = x + cfg.residual_mult * y
            continue
        x = x + y
        h = norm(x, f"l{i}.norm2")
        if f.kind == "experts":
            x = x + _routed(h, w, p, f)
        else:
            u = (h @ w(p + "up").t() + w(p + "up.b")).clamp_(min=0.0).pow(2)
            x = x + u @ w(p + "down").t() + w(p + "down.b")
    return norm(x, "final.norm"), w("embed" if cfg.tied_head else "head")


@torch.no_grad()
def exact(case: dict, seed: int):
    cfg, get = _tensors(case, seed)
    rows = _llama_rows if case["family"] == "llama" else _hybrid_rows

    def w(name):
        return get(name).to(D)
    if case["kind"] == "prompt":
        h, head = rows(cfg, w, torch.tensor(_ids(cfg, case["tokens"], seed), device=DEV))
        return head @ h[-1]
    if case["kind"] == "request":
        ids, n = _ids(cfg, case["tokens"], seed), case["tokens"]
        for _ in range(case["new"]):   # what the head prefers; checked below
            tied = case["family"] == "navalorn"
            ids.append(ids[-1] if tied else (ids[-1] + FOLLOW) % cfg.vocab_size)
        h, head = rows(cfg, w, torch.tensor(ids, device=DEV))
        chosen = []
        for t in range(n - 1, n + case["new"]):
            logits = head @ h[t]
            seen = torch.tensor(sorted(set(ids[max(0, t + 1 - LAST_N):t + 1])), device=DEV)
            s = logits[seen]
            logits[seen] = torch.where(s >= 0, s / PENALTY, s * PENALTY)
            chosen.append(int(logits.argmax()))
        if chosen[:-1] != ids[n:]:
            return None   # a tie after all: the rest of the sequence would be another
        return {"tokens": torch.tensor(chosen), "logits": logits}
    new = case["new"]
    each = []
    for s in _sequences(case, cfg, seed):
        h, head = rows(cfg, w, torch.tensor(s, device=DEV))
        each.append(h[len(s) - new - 1:] @ head.t())
    return [torch.stack([e[k] for e in each]) for k in range(new + 1)]
