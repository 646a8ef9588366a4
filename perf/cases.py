"""The framework's work as a user's program asks for it, for timing and comparison.

A program that uses this framework loads a model once, keeps a KV cache per
session, and then feeds prompts, generates, replays logged sessions (checkout),
steps many sessions in lockstep and, for attribution, exports attention
probabilities and value norms. The cases are those calls, through
``defer_amd.gpu``, on the model shapes of ``defer_amd.synthetic.CONFIGS``
(N(0, 0.02) weights from seed 0, loaded once per process and shape, as a program
that serves a model does). A case's seed makes the sessions: token ids, rng
words and, where the case continues one, the cached history.

``kind`` says what a pass does:

* ``forward``   one token after ``ctx`` cached positions, its logits to the host;
* ``generate``  a turn: ``prompt`` tokens after ``ctx`` cached positions, then
                ``gen`` tokens at ``temp``; tokens and the last logits;
* ``prefill``   ``prompt`` tokens after ``ctx`` cached positions; the last logits;
* ``replay``    checkout of a session of ``prompt`` + ``gen`` tokens sampled at
                ``temp``: every token re-sampled and compared; the last logits;
* ``lockstep``  ``rows`` sessions of about ``ctx`` positions each: a token fed to
                each, ``gen`` steps at ``temp``, then a closing token fed to
                each with its logits to the host;
* ``attribute`` one token after ``ctx`` positions with the attention
                probabilities exported, the value norms of the last ``norms``
                positions, and the same token again with ``mask`` positions
                masked (the ablation).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from defer_amd import gpu as G
from defer_amd import synthetic

DEV = "cuda:0"
SHAPES = ("smollm2-135m", "smollm2-360m", "llama-3.2-1b", "llama-3-8b")


def _case(kind, shape, name=None, **kw):
    c = {"kind": kind, "shape": shape, "ctx": 0, "prompt": 0, "gen": 0, "temp": 0.0, "rows": 1,
         "norms": 0, "mask": 0}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest call: one token of a short session, logits returned.
        _case("forward", "smollm2-135m", "forward-135m", ctx=203),
        # A chat turn: a short user message after some history, a sampled answer.
        _case("generate", "smollm2-135m", "turn-135m", ctx=200, prompt=21, gen=64, temp=0.8),
        # A fresh session on the headline shape: short prompt, greedy answer.
        _case("generate", "smollm2-135m", "greedy-135m", prompt=32, gen=128),
        # Late in a long session: one token fed, a sampled answer.
        _case("generate", "smollm2-360m", "long-360m", ctx=3001, prompt=1, gen=48, temp=0.8),
        # The largest model, one session, greedy.
        _case("generate", "llama-3-8b", "greedy-8b", prompt=64, gen=24),
        # An ordinary prompt.
        _case("prefill", "smollm2-135m", "prefill-135m", prompt=301),
        # A long document as a prompt.
        _case("prefill", "smollm2-360m", "prefill-360m", prompt=3500),
        # A prompt to the largest model.
        _case("prefill", "llama-3-8b", "prefill-8b", prompt=500),
        # Checkout: a logged session verified by re-sampling all of it.
        _case("replay", "smollm2-135m", "replay-135m", prompt=512, gen=1536, temp=0.7),
        # Many sessions stepped together.
        _case("lockstep", "llama-3.2-1b", "lockstep-1b", ctx=256, gen=8, rows=64),
        # A handful of sessions stepped together, sampled.
        _case("lockstep", "smollm2-135m", "lockstep-135m", ctx=150, gen=16, temp=0.8, rows=7),
        # Attribution of one token: trace, value norms, one ablation.
        _case("attribute", "smollm2-135m", "attribute-135m", ctx=400, norms=64, mask=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "generate", "generate", "prefill", "prefill", "prefill", "replay",
                       "lockstep", "lockstep", "attribute"])
    if kind == "forward":
        return _case(kind, rng.choice(SHAPES), ctx=_log_int(rng, 1, 2000))
    if kind == "generate":
        shape = rng.choice(SHAPES)
        big = shape == "llama-3-8b"
        return _case(kind, shape, ctx=rng.choice([0, _log_int(rng, 16, 500 if big else 4000)]),
                     prompt=_log_int(rng, 1, 64 if big else 200),
                     gen=_log_int(rng, 4, {"llama-3-8b": 20, "llama-3.2-1b": 80}.get(shape, 128)),
                     temp=rng.choice([0.0, 0.7, 1.0]))
    if kind == "prefill":
        shape = rng.choice(SHAPES)
        most = {"smollm2-135m": 4000, "smollm2-360m": 3500, "llama-3.2-1b": 2500, "llama-3-8b": 500}[shape]
        return _case(kind, shape, ctx=rng.choice([0, 0, _log_int(rng, 16, 1000 if most > 1000 else 300)]),
                     prompt=_log_int(rng, 16, most))
    if kind == "replay":
        return _case(kind, rng.choice(SHAPES[:2]), prompt=_log_int(rng, 8, 512),
                     gen=_log_int(rng, 32, 1000), temp=rng.choice([0.0, 0.7, 1.0]))
    if kind == "lockstep":
        shape = rng.choice(SHAPES[:3])
        return _case(kind, shape, ctx=_log_int(rng, 16, 500), gen=rng.randint(2, 8),
                     temp=rng.choice([0.0, 0.8]), rows=_log_int(rng, 2, 64))
    return _case(kind, rng.choice(SHAPES[:2]), ctx=_log_int(rng, 70, 1000), norms=_log_int(rng, 8, 64),
                 mask=rng.randint(1, 32))


_LOADED = {}  # the one model this process holds: shape -> GpuModel


def _model(shape):
    if shape not in _LOADED:
        _LOADED.clear()  # a model goes with its last cache
        cfg = synthetic.CONFIGS[shape]
        _LOADED[shape] = G.GpuModel(G.Config.from_dict(cfg), synthetic.make_weights(cfg, 0, threads=16))
    return _LOADED[shape]


def _tokens(case, seed):
    """Token ids and rng words of every session of the case, from the seed alone."""
    cfg = synthetic.CONFIGS[case["shape"]]
    g = np.random.Generator(np.random.PCG64(seed))
    V, n = cfg["vocab_size"], case["rows"]
    # sessions in lockstep have lengths of their own
    ctx = [case["ctx"]] if n == 1 else [max(1, int(case["ctx"] * g.uniform(0.5, 1.5))) for _ in range(n)]
    return {
        "hist": [g.integers(0, V, size=k, dtype=np.uint32) for k in ctx],
        "prompt": g.integers(0, V, size=case["prompt"], dtype=np.uint32),
        "feed": g.integers(0, V, size=(2, n), dtype=np.uint32),
        "words": g.integers(0, 1 << 32, size=(max(case["gen"], 1), n), dtype=np.uint32),
        "mask": g.permutation(case["ctx"])[: case["mask"]].astype(np.uint32),
    }


def prepare(case, seed):
    m = _model(case["shape"])
    s = dict(_tokens(case, seed), case=case, model=m)
    room = case["prompt"] + case["gen"] + 4
    s["caches"] = []
    for h in s["hist"]:
        c = m.new_cache(len(h) + room)
        if len(h):
            m.prompt(c, h)
        s["caches"].append(c)
    if case["kind"] == "replay":  # the logged session: what this model sampled
        c = s["caches"][0]
        m.prompt(c, s["prompt"])
        words = s["words"][:, 0]
        out = m.generate(c, case["gen"], case["temp"], words)
        s["log"] = np.concatenate([s["prompt"], np.asarray(out, dtype=np.uint32)])
    return s


def run(s):
    case, m, c = s["case"], s["model"], s["caches"][0]
    kind, T = case["kind"], case["temp"]
    words = s["words"]
    if kind == "lockstep":
        cs = s["caches"]
        for x, h in zip(cs, s["hist"]):
            x.truncate(len(h))
        m.forward_batch(cs, s["feed"][0])
        toks = [m.step_batch(cs, T, words[i] if T else None) for i in range(case["gen"])]
        logits = m.forward_batch(cs, s["feed"][1], logits=True)
        return {"tokens": np.asarray(toks, dtype=np.int64), "logits": logits}
    c.truncate(len(s["hist"][0]))
    if kind == "forward":
        return {"logits": m.forward(int(s["feed"][0, 0]), c)}
    if kind == "generate":
        m.prompt(c, s["prompt"])
        toks = m.generate(c, case["gen"], T, words[:, 0] if T else None)
        return {"tokens": np.asarray(toks, dtype=np.int64), "logits": c.last_logits()}
    if kind == "prefill":
        m.prompt(c, s["prompt"])
        return {"logits": c.last_logits()}
    if kind == "replay":
        div, _ = m.replay(c, s["log"], case["prompt"], T, words[:, 0] if T else None)
        return {"first_divergence": div, "logits": c.last_logits()}
    tok = int(s["feed"][0, 0])
    logits, probs = m.forward(tok, c, trace=True)
    n = len(c)
    norms = c.value_norms(n - case["norms"], n)
    c.truncate(n - 1)
    masked = m.forward(tok, c, masked=s["mask"])
    return {"logits": logits, "probs": probs, "norms": norms, "masked_logits": masked}


def work(case):
    """Bytes: the f32 weights once per step that needs them (a prompt or a
    batch step streams them once), the cached K/V read and written, logits out.
    Flops: two per weight and row, plus attention's scores and values."""
    cfg = synthetic.CONFIGS[case["shape"]]
    h, V, ff, L = cfg["hidden_size"], cfg["vocab_size"], cfg["intermediate_size"], cfg["num_layers"]
    q, kv = cfg["num_heads"] * cfg["head_dim"], cfg["num_kv_heads"] * cfg["head_dim"]
    layers = 4 * L * ((q + 2 * kv) * h + h * q + 3 * ff * h)  # bytes of the layers' matrices
    head = 4 * V * h
    kvb = 8 * L * kv  # K and V bytes of one position
    total = {"bytes": 0.0, "flops": 0.0}

    def step(rows, read, heads, fresh):
        # rows fed together; read: cached positions read (each once per
        # session); heads: rows whose logits are formed; fresh: sum over the
        # rows of the positions each attends to
        total["bytes"] += layers + (head if heads else 0) + kvb * (read + rows) + 4 * V * heads
        total["flops"] += layers / 2 * rows + head / 2 * heads + 4 * L * q * fresh

    def tri(a, n):  # positions attended by n rows after a cached ones
        return n * a + n * (n + 1) / 2

    ctx, p, g, n = case["ctx"], case["prompt"], case["gen"], case["rows"]
    kind = case["kind"]
    if kind == "forward":
        step(1, ctx, 1, ctx + 1)
    elif kind in ("generate", "prefill"):
        step(p, ctx, 1, tri(ctx, p))
        for i in range(g):
            step(1, ctx + p + i, 1, ctx + p + i + 1)
    elif kind == "replay":
        step(p + g, 0, g + 1, tri(0, p + g))
    elif kind == "lockstep":
        for i in range(g + 2):
            step(n, n * (ctx + i), n, n * (ctx + i + 1))
    else:
        step(1, ctx, 1, ctx + 1)
        step(1, ctx, 1, ctx + 1 - case["mask"])
        heads = cfg["num_heads"]
        total["bytes"] += 4 * L * (heads * (ctx + 1) + h * q + case["norms"] * (kv + heads))
        total["flops"] += 2 * L * h * q * case["norms"]
    return total


def tolerance(case):
    """Everything is f32, every sum a chain or tree of f32 terms. The logits'
    error against 64 bits (what another order of the same sums shows as well)
    grows with depth and width: 4e-7 measured on the 135M shape, 7e-7 on 360M,
    2.3e-6 on 1B, 7e-6 on 8B; stated at about four times that. Tokens are
    compared whole."""
    rel = {"smollm2-135m": 2e-6, "smollm2-360m": 3e-6, "llama-3.2-1b": 1e-5, "llama-3-8b": 3e-5}
    return {"rel": rel[case["shape"]], "max": 20 * rel[case["shape"]], "differ": 0.0}


# ------------------------------------------------- the same in 64 bits


class _Exact:
    """The model in float64, plain torch, weights on the GPU."""

    def __init__(self, shape):
        self.cfg = cfg = synthetic.CONFIGS[shape]
        it = iter(synthetic.make_weights(cfg, 0, threads=16))
        keep = torch.float64 if shape != "llama-3-8b" else torch.float32  # widened where used
        up = lambda: torch.from_numpy(next(it)).to(DEV).to(keep)  # noqa: E731
        self.embed = up()
        names = ("n1", "wq", "wk", "wv", "wo", "n2", "wg", "wu", "wd")
        self.layers = [{k: up() for k in names} for _ in range(cfg["num_layers"])]
        self.norm = up()
        self.head = self.embed if cfg["tie_word_embeddings"] else up()
        half = cfg["head_dim"] // 2
        inv = 1.0 / cfg["rope_theta"] ** (torch.arange(half, dtype=torch.float64, device=DEV) * 2 / cfg["head_dim"])
        # the angles are float32 by definition: position times the float32 frequency
        ang = torch.arange(cfg["max_seq_len"], dtype=torch.float32, device=DEV)[:, None] * inv.float()[None]
        self.cos, self.sin = ang.double().cos(), ang.double().sin()

    def _norm(self, x, w):
        return x / (x.square().mean(-1, keepdim=True) + self.cfg["rms_norm_eps"]).sqrt() * w.double()

    def _rope(self, x, pos):  # [n, heads, hd]
        a, b = x.chunk(2, -1)
        c, s = self.cos[pos][:, None], self.sin[pos][:, None]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    def feed(self, caches, counts, tokens, masked=None, probs=None):
        """counts[i] tokens to caches[i] (a list per layer of [K, V]); the hidden rows."""
        cfg = self.cfg
        nh, nkv, hd = cfg["num_heads"], cfg["num_kv_heads"], cfg["head_dim"]
        at = [0 if c[0] is None else c[0][0].shape[0] for c in caches]
        pos = torch.cat([torch.arange(a, a + k, device=DEV) for a, k in zip(at, counts)])
        x = self.embed[torch.as_tensor(np.asarray(tokens, dtype=np.int64), device=DEV)].double()
        for li, W in enumerate(self.layers):
            y = self._norm(x, W["n1"])
            q = self._rope((y @ W["wq"].double().T).view(-1, nh, hd), pos)
            k = self._rope((y @ W["wk"].double().T).view(-1, nkv, hd), pos)
            v = (y @ W["wv"].double().T).view(-1, nkv, hd)
            out, o = [], 0
            for c, a, n in zip(caches, at, counts):
                if c[li] is not None:
                    K, Vv = torch.cat([c[li][0], k[o:o + n]]), torch.cat([c[li][1], v[o:o + n]])
                else:
                    K, Vv = k[o:o + n], v[o:o + n]
                c[li] = (K, Vv)
                hide = torch.arange(a + n, device=DEV)[None] > torch.arange(a, a + n, device=DEV)[:, None]
                if masked is not None:
                    hide[:, torch.as_tensor(np.asarray(masked, dtype=np.int64), device=DEV)] = True
                heads, P = [], []
                for g in range(nkv):
                    for j in range(nh // nkv):
                        sc = q[o:o + n, g * (nh // nkv) + j] @ K[:, g].T.contiguous() / math.sqrt(hd)
                        pr = torch.softmax(sc.masked_fill(hide, -math.inf), -1)
                        heads.append(pr @ Vv[:, g].contiguous())
                        P.append(pr[-1])
                if probs is not None:
                    probs.append(torch.stack(P))
                out.append(torch.cat(heads, -1))
                o += n
            x = x + torch.cat(out) @ W["wo"].double().T
            y = self._norm(x, W["n2"])
            x = x + (torch.nn.functional.silu(y @ W["wg"].double().T) * (y @ W["wu"].double().T)) @ W["wd"].double().T
        return x

    def logits(self, x):
        y = self._norm(x, self.norm)
        return torch.cat([y @ w.double().T for w in self.head.split(16384)], -1)

    def new(self):
        return [None] * self.cfg["num_layers"]


_EXACT = {}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("generate", "lockstep") and case["temp"]:
        return None  # a draw next to an edge of the CDF is decided by rounding, and all that follows with it
    if kind == "replay":
        return None  # the log is what the f32 model sampled
    if case["shape"] not in _EXACT:
        _EXACT.clear()
        torch.cuda.empty_cache()
        _EXACT[case["shape"]] = _Exact(case["shape"])
    E, t = _EXACT[case["shape"]], _tokens(case, seed)
    with torch.no_grad():
        caches = [E.new() for _ in t["hist"]]
        for c, h in zip(caches, t["hist"]):
            if len(h):
                E.feed([c], [len(h)], h)
        one = [1] * len(caches)
        if kind == "lockstep":
            x, toks = E.feed(caches, one, t["feed"][0]), []
            for _ in range(case["gen"]):
                toks.append(E.logits(x).argmax(-1).cpu().numpy())
                x = E.feed(caches, one, toks[-1])
            return {"tokens": None, "logits": E.logits(E.feed(caches, one, t["feed"][1])).cpu().numpy()}
        if kind == "attribute":
            probs, tok = [], t["feed"][0, :1]
            old = [list(c) for c in caches]
            x = E.feed(caches, one, tok, probs=probs)
            cfg, n = E.cfg, case["ctx"] + 1
            nh, grp, hd = cfg["num_heads"], cfg["num_heads"] // cfg["num_kv_heads"], cfg["head_dim"]
            norms = [torch.stack([(caches[0][li][1][n - case["norms"]:, hh // grp] @
                                   W["wo"].double()[:, hh * hd:(hh + 1) * hd].T.contiguous()).norm(dim=-1)
                                  for hh in range(nh)], -1) for li, W in enumerate(E.layers)]
            y = E.feed(old, one, tok, masked=t["mask"])
            return {"logits": E.logits(x)[0].cpu().numpy(), "probs": torch.stack(probs).cpu().numpy(),
                    "norms": torch.stack(norms).cpu().numpy(), "masked_logits": E.logits(y)[0].cpu().numpy()}
        x = E.feed(caches, [1], t["feed"][0, :1]) if kind == "forward" else E.feed(caches, [case["prompt"]], t["prompt"])
        for _ in range(case["gen"]):
            x = E.feed(caches, [1], [int(E.logits(x[-1:]).argmax())])
        out = {"logits": E.logits(x[-1:])[0].cpu().numpy()}
        return {"tokens": None, **out} if kind == "generate" else out
