"""What the framework's speed is measured on: the work that its users have it do, through its public entry points.

``listed()`` names the cases, ``draw(rng)`` gives another one of the same ranges.  Of a case, ``prepare`` makes what a program
has in hand before the call (a model on the GPU, requests whose prompts are cached, the tokens that come next), ``run`` is one
pass, ``exact`` the same outputs in 64 bits from plain torch, ``work`` what a pass cannot do without, and ``tolerance`` how far
two correct implementations are apart.

Kinds of pass:

========  ==========================================================================================================
decode    one step of single tokens for ``batch`` requests with up to ``context`` cached tokens each (half of it at least);
          a request grows by a token a pass, as it does in earnest
prompt    a prompt of ``tokens`` tokens in portions of 2,048 (the scheduler's budget), up to the logits of its last position,
          or with ``score`` of all its positions (perplexities, comparing a model's logits)
mixed     one step that carries ``tokens`` tokens of a prompt beside ``batch`` decoded tokens
replay    a trace replayed as the replay tool does it: prompts in one step, then ``new`` steps of given tokens, every step's
          logits on the host
sample    picking the next token of ``rows`` rows of logits with temperature and cuts
========  ==========================================================================================================

Models are the shapes of this repository's benchmark at their real layer sizes.  They have eight layers (the 1B class its 16,
Suripel one period of six): what a layer costs is the same, and a state is made quickly.  Weights are random: matrices
N(0, 0.02), those that write to the residual stream smaller by sqrt(2 layers), the embedding N(0, 1), so that the stream
changes by a fraction a layer as it does in a trained model.  (With N(0, 0.02) everywhere the first layer's result is seventy
times the embedding, every later layer amplifies its rounding errors, and two correct bfloat16 implementations are 2-3% apart.)
"""
from __future__ import annotations

import math
from typing import Any, Dict, List

import numpy as np
import torch

PORTION = 2048      # tokens of a prompt a step takes
ROOM = 4096         # tokens that a decoding request may grow by before it is begun again

_LLAMA3 = {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
           "original_max_position_embeddings": 8192}


def _llama(layers, hidden, heads, kv_heads, head_dim, inter, vocab, theta=500000.0, scaling=None, tied=False, context=16384) -> dict:
    return {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "num_hidden_layers": layers, "hidden_size": hidden,
            "num_attention_heads": heads, "num_key_value_heads": kv_heads, "head_dim": head_dim, "intermediate_size": inter,
            "vocab_size": vocab, "rope_theta": theta, "rms_norm_eps": 1e-5, "tie_word_embeddings": tied,
            "max_position_embeddings": context, "hidden_act": "silu", **({"rope_scaling": scaling} if scaling else {})}


def _suripel(width) -> dict:
    """One period of the benchmark's Suripel layers: retention, windowed attention with block means, the gated delta rule, an
    attention that reads the first one's keys and values, retention, the delta rule; a dense PolyNorm feed-forward."""
    heads = width // 128
    ff = {"kind": "dense", "ff": int(width * 5.25)}
    att = {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 128, "vdim": 128, "conv": 4, "scale": 128 ** -0.5,
           "mask": {"size": 1024, "pool": 64}}
    delta = {"type": "delta", "mixer": {"heads": heads, "kv_heads": max(1, heads // 2), "dim": 128, "vdim": 128, "conv": 4}, "mlp": ff}
    ret = {"type": "retention", "mlp": ff,
           "mixer": {"heads": heads, "dim": 128, "vdim": 128, "decay": [1 - 0.06 * 0.75 ** (8 * i / heads) for i in range(heads)],
                     "rot": {"dims": 128, "base": 1e6}}}
    layers = [ret, {"type": "attention", "mixer": att, "mlp": ff}, delta, {"type": "attention", "mixer": dict(att, kv_from=1), "mlp": ff},
              ret, delta]
    return {"architecture": "Suripel", "vocab": 32000, "width": width, "norm": {"eps": 1e-5}, "canon": {"taps": 4}, "layers": layers}


MODELS = {
    "tiny": _llama(2, 64, 4, 2, 16, 176, 256, theta=10000.0, context=128),
    "llama-1b-head64": _llama(16, 2048, 32, 8, 64, 8192, 128256, scaling=dict(_LLAMA3, factor=32.0), tied=True),
    "llama-3.1-8b": _llama(8, 4096, 32, 8, 128, 14336, 128256, scaling=_LLAMA3),
    "llama-2-7b": _llama(8, 4096, 32, 32, 128, 11008, 32000, theta=10000.0),
    "suripel-2048": _suripel(2048),
    "suripel-4096": _suripel(4096),
}


# ------------------------------------------------------------------------------------------------ the cases
def listed() -> List[Dict[str, Any]]:
    return [
        # a test's or a debugging session's trace on the tiny model, in true 32 bits: nothing but launches and the host
        {"name": "replay-tiny-f32", "kind": "replay", "model": "tiny", "dtype": "float32", "requests": 3, "tokens": 33, "new": 16},
        # one user at a time on a small model: the lowest latency a token can have
        {"name": "decode-1b-b1", "kind": "decode", "model": "llama-1b-head64", "dtype": "bfloat16", "batch": 1, "context": 700},
        # one user, ordinary model
        {"name": "decode-8b-b1", "kind": "decode", "model": "llama-3.1-8b", "dtype": "bfloat16", "batch": 1, "context": 1900},
        # a small server: the benchmark's own point
        {"name": "decode-8b-b8", "kind": "decode", "model": "llama-3.1-8b", "dtype": "bfloat16", "batch": 8, "context": 2000},
        # a busy server, requests of all lengths
        {"name": "decode-8b-b64", "kind": "decode", "model": "llama-3.1-8b", "dtype": "bfloat16", "batch": 64, "context": 1900},
        # a question typed by hand: time to the first token
        {"name": "prompt-8b-137", "kind": "prompt", "model": "llama-3.1-8b", "dtype": "bfloat16", "tokens": 137, "score": False},
        # a document, in the scheduler's portions
        {"name": "prompt-8b-5000", "kind": "prompt", "model": "llama-3.1-8b", "dtype": "bfloat16", "tokens": 5000, "score": False},
        # continuous batching: a portion of somebody's prompt beside everybody's next token
        {"name": "mixed-7b", "kind": "mixed", "model": "llama-2-7b", "dtype": "bfloat16", "tokens": 1501, "batch": 23, "context": 900},
        # the true 32-bit path over a text, all positions' logits: what a bfloat16 model is held against
        {"name": "score-1b-f32", "kind": "prompt", "model": "llama-1b-head64", "dtype": "float32", "tokens": 401, "score": True},
        # chat sampling for a busy server
        {"name": "sample-b64", "kind": "sample", "rows": 64, "vocab": 128256, "temperature": 0.8, "top_k": 0, "top_p": 0.95,
         "min_p": 0.0, "repeat_penalty": 1.0},
        # the other kind of decoder: recurrences, short convolutions, windowed attention
        {"name": "prompt-suripel-2048", "kind": "prompt", "model": "suripel-4096", "dtype": "bfloat16", "tokens": 2048, "score": False},
        {"name": "decode-suripel-b8", "kind": "decode", "model": "suripel-2048", "dtype": "bfloat16", "batch": 8, "context": 1900},
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> Dict[str, Any]:
    kind = rng.choice(["decode"] * 4 + ["prompt"] * 4 + ["mixed", "replay", "sample", "sample"])
    if kind == "decode":
        model = rng.choice(["llama-3.1-8b", "llama-3.1-8b", "llama-1b-head64", "llama-2-7b", "suripel-2048", "suripel-4096"])
        batch = _log(rng, 1, 64)
        # (as many cached tokens at most as the largest listed case has: heads that are not grouped keep four times as many bytes)
        most = 110000 // (4 if model == "llama-2-7b" else 1)
        return {"kind": kind, "model": model, "dtype": "bfloat16", "batch": batch, "context": _log(rng, 64, min(8000, most // batch))}
    if kind == "prompt":
        model = rng.choice(["llama-3.1-8b", "llama-3.1-8b", "llama-1b-head64", "llama-2-7b", "suripel-2048", "suripel-4096"])
        if rng.random() < 0.25:
            return {"kind": kind, "model": rng.choice(["tiny", "llama-1b-head64"]), "dtype": "float32", "tokens": _log(rng, 8, 128), "score": True}
        return {"kind": kind, "model": model, "dtype": "bfloat16",
                "tokens": _log(rng, 16, 2048 if model.startswith("suripel") else 4500), "score": False}
    if kind == "mixed":
        return {"kind": kind, "model": rng.choice(["llama-3.1-8b", "llama-2-7b"]), "dtype": "bfloat16", "tokens": _log(rng, 32, 1600),
                "batch": _log(rng, 2, 40), "context": _log(rng, 64, 1000)}
    if kind == "replay":
        return {"kind": kind, "model": "tiny", "dtype": rng.choice(["float32", "bfloat16"]), "requests": rng.randint(1, 4),
                "tokens": rng.randint(1, 64), "new": rng.randint(4, 24)}
    return {"kind": kind, "rows": _log(rng, 1, 64), "vocab": rng.choice([32000, 128256]), "temperature": round(rng.uniform(0.3, 1.3), 2),
            "top_k": rng.choice([0, 0, 20, 40, 200]), "top_p": rng.choice([1.0, 0.8, 0.9, 0.95]), "min_p": rng.choice([0.0, 0.0, 0.05]),
            "repeat_penalty": rng.choice([1.0, 1.0, 1.1])}


# ------------------------------------------------------------------------------------------------ inputs
def _tokens(seed: int, vocab: int, *shape) -> np.ndarray:
    return np.random.default_rng(seed).integers(0, vocab, size=shape)


def _weights(cfg: dict, dtype: str, seed: int) -> Dict[str, torch.Tensor]:
    """The model's tensors by name, on the GPU, in the storage type of ``dtype``."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 2 + 1)
    dt = getattr(torch, dtype)
    out: Dict[str, torch.Tensor] = {}

    def matrix(name, *shape, std=0.02, mean=0.0):
        out[name] = (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std + mean).to(dt)

    def ones(name, n):
        out[name] = torch.ones((n,), device="cuda", dtype=dt)

    write = 0.02 / math.sqrt(2 * (len(cfg["layers"]) if "layers" in cfg else cfg["num_hidden_layers"]))
    if cfg.get("architecture") == "Suripel":
        E = cfg["width"]
        matrix("embed", cfg["vocab"], E, std=1.0)
        for i, layer in enumerate(cfg["layers"]):
            p, m, kind = f"l{i}.", layer["mixer"], layer["type"]
            H, D, Dv = m["heads"], m["dim"], m["vdim"]
            G = m.get("kv_heads", H)
            ones(p + "norm1", E), ones(p + "norm2", E)
            matrix(p + "canon1", E, 4, std=0.2), matrix(p + "canon2", E, 4, std=0.2)
            own = kind != "attention" or "kv_from" not in m
            sizes = {"q": (G if kind == "delta" else H) * D}
            if own:
                sizes.update(k=G * D, v=(H if kind == "delta" else G) * Dv)
            for name, n in sizes.items():
                matrix(p + "mix." + name, n, E)
                if "conv" in m:
                    matrix(p + "mix." + name + ".conv", n, m["conv"], std=0.2, mean=0.25)
            if kind != "attention":
                matrix(p + "mix.g", H * Dv, E)
            if kind == "delta":
                matrix(p + "mix.a", H, E), matrix(p + "mix.b", H, E)
                matrix(p + "mix.A_log", H, std=0.3), matrix(p + "mix.dt_bias", H, std=0.3, mean=-3.0)
                ones(p + "mix.norm", Dv)
            matrix(p + "mix.o", E, H * Dv, std=write)
            F = layer["mlp"]["ff"]
            matrix(p + "mlp.up", F, E), matrix(p + "mlp.down", E, F, std=write)
            out[p + "mlp.act"] = torch.tensor([1 / 3, 1 / 3, 1 / 3, 0.0], device="cuda").to(dt)
        ones("final.norm", E)
        matrix("head", cfg["vocab"], E)
        return out
    E, H, G, D, F = (cfg[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim", "intermediate_size"))
    matrix("model.embed_tokens.weight", cfg["vocab_size"], E, std=1.0)
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        ones(p + "input_layernorm.weight", E), ones(p + "post_attention_layernorm.weight", E)
        for name, n, k in (("self_attn.q_proj", H * D, E), ("self_attn.k_proj", G * D, E), ("self_attn.v_proj", G * D, E),
                           ("self_attn.o_proj", E, H * D), ("mlp.gate_proj", F, E), ("mlp.up_proj", F, E), ("mlp.down_proj", E, F)):
            matrix(p + name + ".weight", n, k, std=write if name in ("self_attn.o_proj", "mlp.down_proj") else 0.02)
    ones("model.norm.weight", E)
    if not cfg["tie_word_embeddings"]:
        matrix("lm_head.weight", cfg["vocab_size"], E)
    return out


def _vocab(cfg: dict) -> int:
    return cfg.get("vocab_size") or cfg["vocab"]


def _contexts(case, seed) -> List[int]:
    """Cached tokens of every decoding request: the longest as long as the case says, the others half of that at least."""
    n = np.random.default_rng(seed + 7).integers(max(1, case["context"] // 2), case["context"] + 1, size=case["batch"])
    n[0] = case["context"]
    return [int(x) for x in n]


def _cached(case, seed) -> List[np.ndarray]:
    """The prompts of the decoding requests."""
    vocab = _vocab(MODELS[case["model"]])
    return [_tokens(seed * 1000 + 17 + i, vocab, n) for i, n in enumerate(_contexts(case, seed))]


def _replay_lengths(case, seed) -> List[int]:
    n = case["requests"]
    return [max(1, case["tokens"] * (i + 1) // n) for i in range(n)]


# ------------------------------------------------------------------------------------------------ a pass
def _runner(case, seed, max_tokens, max_requests):
    from xyntetik_runner_amd.config import config_from_dict
    from xyntetik_runner_amd.engine import ModelRunner
    cfg = MODELS[case["model"]]
    arch, typed = config_from_dict(cfg)
    return ModelRunner(arch.build_spec(typed), _weights(cfg, case["dtype"], seed), case["dtype"], max_tokens=max_tokens,
                       page_size=64, max_requests=max_requests, consume_state=True)


def _cache_prompts(s) -> None:
    """The decoding requests from their start: prompts into the cache, and the first decoded token, as a server would have run them."""
    r, Entry = s["runner"], s["entry"]
    for i, toks in enumerate(s["cached"]):
        if r.has(i):
            r.finish(i)
        for a in range(0, len(toks), PORTION):
            r.step([Entry(i, toks[a:a + PORTION], [])])
    s["at"] = 0
    if s["kind"] == "decode":
        _decode_step(s)


def _decode_step(s):
    toks = s["next"][s["at"]]
    s["at"] += 1
    return s["runner"].step([s["entry"](i, [t], [0]) for i, t in enumerate(toks)])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sample":
        from xyntetik_runner_amd.csrc.ops import load_ops
        from xyntetik_runner_amd.sampling import Sampler, SamplerState, SamplingParams
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        logits = torch.randn((case["rows"], case["vocab"]), generator=g, device="cuda") * 2.5
        states = []
        for r in range(case["rows"]):
            st = SamplerState(SamplingParams(temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"], min_p=case["min_p"],
                                             repeat_penalty=case["repeat_penalty"], seed=seed * 131 + r + 1))
            for t in _tokens(seed * 1000 + r, case["vocab"], 300).tolist():
                st.accept(t)
            states.append(st)
        return {"kind": kind, "sampler": Sampler(load_ops(), torch.device("cuda:0")), "logits": logits, "states": states}
    from xyntetik_runner_amd.engine.batch import StepEntry
    cfg = MODELS[case["model"]]
    vocab = _vocab(cfg)
    s: Dict[str, Any] = {"kind": kind, "entry": StepEntry}
    if kind in ("decode", "mixed"):
        cached = _cached(case, seed)
        span = sum(-(-(len(t) + ROOM) // 64) * 64 for t in cached) + (-(-case["tokens"] // 64) * 64 if kind == "mixed" else 0)
        s.update(runner=_runner(case, seed, span, case["batch"] + 1), cached=[t.tolist() for t in cached],
                 next=_tokens(seed + 3, vocab, ROOM, case["batch"]).tolist())
        if kind == "mixed":
            s["prompt"] = _tokens(seed + 5, vocab, case["tokens"]).tolist()
        _cache_prompts(s)
    elif kind == "prompt":
        s.update(runner=_runner(case, seed, -(-case["tokens"] // 64) * 64, 1), prompt=_tokens(seed + 5, vocab, case["tokens"]).tolist(),
                 score=case["score"])
    else:
        lens = _replay_lengths(case, seed)
        s.update(runner=_runner(case, seed, sum(-(-(n + case["new"]) // 64) * 64 for n in lens), len(lens)),
                 prompts=[_tokens(seed * 1000 + 17 + i, vocab, n).tolist() for i, n in enumerate(lens)],
                 next=_tokens(seed + 3, vocab, case["new"], len(lens)).tolist())
    return s


def run(s):
    kind = s["kind"]
    if kind == "sample":
        return s["sampler"].launch(s["logits"], s["states"])
    r, Entry = s["runner"], s["entry"]
    if kind == "decode":
        if s["at"] >= ROOM - 1:
            _cache_prompts(s)
        return _decode_step(s)
    if kind == "mixed":
        if s["at"] >= ROOM - 1:
            _cache_prompts(s)
        n = len(s["prompt"])
        toks = s["next"][s["at"]]
        s["at"] += 1
        out = r.step([Entry("new", s["prompt"], [n - 1])] + [Entry(i, [t], [0]) for i, t in enumerate(toks)])
        r.finish("new")
        return out
    if kind == "prompt":
        toks, out = s["prompt"], []
        for a in range(0, len(toks), PORTION):
            part = toks[a:a + PORTION]
            last = a + len(part) == len(toks)
            got = r.step([Entry("p", part, list(range(len(part))) if s["score"] else [len(part) - 1] if last else [])])
            if got is not None:
                out.append(got)
        r.finish("p")
        return out
    # replay: every step's logits go to the host before the next step is read
    out = [r.step([Entry(i, t, [len(t) - 1]) for i, t in enumerate(s["prompts"])]).cpu()]
    for toks in s["next"]:
        out.append(r.step([Entry(i, [t], [0]) for i, t in enumerate(toks)]).cpu())
    for i in range(len(s["prompts"])):
        r.finish(i)
    return out


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _parameters(cfg) -> int:
    """Weights of the layers (not the embedding, not the head)."""
    if cfg.get("architecture") == "Suripel":
        E, n = cfg["width"], 0
        for layer in cfg["layers"]:
            m = layer["mixer"]
            H, D, Dv = m["heads"], m["dim"], m["vdim"]
            G = m.get("kv_heads", H)
            n += 2 * E * layer["mlp"]["ff"] + E * H * Dv
            if layer["type"] == "attention":
                n += E * (H * D + (0 if "kv_from" in m else G * (D + Dv)))
            elif layer["type"] == "delta":
                n += E * (2 * G * D + 2 * H * Dv + 2 * H)
            else:
                n += E * (2 * H * D + 2 * H * Dv)
        return n
    E, H, G, D, F = (cfg[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim", "intermediate_size"))
    return cfg["num_hidden_layers"] * (2 * E * H * D + 2 * E * G * D + 3 * E * F)


def _cache_row(cfg) -> int:
    """Values a cached token holds, and (second) the products a query does with a key and its value, over all layers."""
    if cfg.get("architecture") == "Suripel":
        att = [l["mixer"] for l in cfg["layers"] if l["type"] == "attention"]
        return sum(m["kv_heads"] * (m["dim"] + m["vdim"]) for m in att), sum(m["heads"] * (m["dim"] + m["vdim"]) for m in att)
    L, D = cfg["num_hidden_layers"], cfg["head_dim"]
    return 2 * L * cfg["num_key_value_heads"] * D, 2 * L * cfg["num_attention_heads"] * D


def work(case) -> Dict[str, float]:
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": 4.0 * case["rows"] * case["vocab"], "flops": 0.0}
    cfg = MODELS[case["model"]]
    elt = 4 if case["dtype"] == "float32" else 2
    suripel = cfg.get("architecture") == "Suripel"
    E, V = cfg.get("hidden_size") or cfg["width"], _vocab(cfg)
    body, (row, pair) = _parameters(cfg), _cache_row(cfg)
    window = 1024 + 128 if suripel else 1 << 30     # (a query reads the window's keys and a mean a block behind it)
    state = sum(m["mixer"]["heads"] * m["mixer"]["dim"] * m["mixer"]["vdim"] for m in cfg["layers"] if m["type"] != "attention") if suripel else 0

    def step(new, seqs, wanted):
        """One step: ``new`` tokens over ``seqs`` (cached, new) pairs, ``wanted`` rows of logits."""
        keys = sum(min(c + n, window + n) for c, n in seqs)
        pairs = sum(min(c, window) * n + min(n, window) * (n - min(n, window) / 2) for c, n in seqs)
        weights = body + (V * E if wanted else 0)
        return np.array([elt * (weights + new * E + row * keys) + 8.0 * state * len(seqs) + 4.0 * wanted * V,
                         2.0 * body * new + 2.0 * V * E * wanted + 2.0 * pair * pairs + 6.0 * state * new])

    if kind == "decode":
        got = step(case["batch"], [(3 * case["context"] // 4, 1)] * case["batch"], case["batch"])
    elif kind == "mixed":
        got = step(case["batch"] + case["tokens"], [(3 * case["context"] // 4, 1)] * case["batch"] + [(0, case["tokens"])], case["batch"] + 1)
    elif kind == "prompt":
        got, n = np.zeros(2), case["tokens"]
        for a in range(0, n, PORTION):
            k = min(PORTION, n - a)
            got = got + step(k, [(a, k)], k if case["score"] else int(a + k == n))
    else:
        lens = _replay_lengths(case, 0)
        got = step(sum(lens), [(0, n) for n in lens], len(lens))
        for i in range(case["new"]):
            got = got + step(len(lens), [(n + i, 1) for n in lens], len(lens))
    return {"bytes": float(got[0]), "flops": float(got[1])}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"      # masses are whole numbers and every cut is defined: the token is too
    # measured against ``exact``: 1e-7 to 4e-7 in 32 bits, 0.0023 to 0.0053 in bfloat16
    if case["dtype"] == "float32":
        return {"rel": 2e-6, "max": 5e-5}
    return {"rel": 0.02, "max": 0.2}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def _mm(x, w, rows=16384):
    """``x w^T`` in 64 bits, some rows at a time."""
    w = w.double()
    return torch.cat([x[a:a + rows] @ w.T for a in range(0, x.shape[0], rows)])


def _rotate(x, positions, inv_freq):
    """Channel j of every head of ``x [T, H, D]`` turned with channel j + D/2 by a 32-bit product of position and frequency."""
    a = (positions.float()[:, None] * inv_freq.float()[None, :]).double()
    c, s = a.cos()[:, None, :], a.sin()[:, None, :]
    u, v = x.chunk(2, dim=-1)
    return torch.cat([u * c - v * s, v * c + u * s], dim=-1)


def _inv_freq(dims, theta, scaling=None):
    inv = float(theta) ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device="cuda") / dims)
    if not scaling:
        return inv
    wave, orig = 2 * math.pi / inv, scaling["original_max_position_embeddings"]
    low, high, factor = scaling["low_freq_factor"], scaling["high_freq_factor"], scaling["factor"]
    mix = ((orig / wave - low) / (high - low)).clamp(0.0, 1.0)
    return (1 - mix) * inv / factor + mix * inv


def _attend(q, k, v, scale, window=None, pool=0):
    """Causal attention of one sequence, ``q [T, H, D]`` over ``k, v [T, G, D]``; with ``pool`` also the mean key and value of every
    block of that many positions that lies wholly behind the window."""
    T, H, D = q.shape
    G = k.shape[1]
    out = torch.empty((T, H, v.shape[2]), dtype=q.dtype, device=q.device)
    n = T // pool if pool else 0
    if n:
        mk, mv = (x[:n * pool].reshape(n, pool, G, -1).mean(1) for x in (k, v))
        end = torch.arange(n, device=q.device) * pool + pool - 1
    for a in range(0, T, 1024):
        b = min(T, a + 1024)
        lo = max(0, a - window + 1) if window else 0
        i, j = torch.arange(a, b, device=q.device)[:, None], torch.arange(lo, b, device=q.device)[None, :]
        see = (j <= i) & ((j > i - window) if window else True)
        if n:
            see = torch.cat([see, end[None, :] <= i - window], dim=1)
        for g in range(G):
            kk, vv = k[lo:b, g], v[lo:b, g]
            if n:
                kk, vv = torch.cat([kk, mk[:, g]]), torch.cat([vv, mv[:, g]])
            for h in range(g * (H // G), (g + 1) * (H // G)):
                s = (q[a:b, h] @ kk.T * scale).masked_fill(~see, float("-inf"))
                out[a:b, h] = torch.softmax(s, dim=-1) @ vv
    return out


def _each(seqs, fn, *xs):
    """``fn`` of every sequence's rows of ``xs``, one after another."""
    out, a = [], 0
    for n in seqs:
        out.append(fn(*(x[a:a + n] for x in xs)))
        a += n
    return torch.cat(out)


def _exact_llama(cfg, w, seqs):
    E, H, G, D = (cfg[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim"))
    lens = [len(t) for t in seqs]
    x = w["model.embed_tokens.weight"][torch.as_tensor(np.concatenate(seqs), device="cuda")].double()
    pos = torch.cat([torch.arange(n, device="cuda") for n in lens])
    freq = _inv_freq(D, cfg["rope_theta"], cfg.get("rope_scaling"))

    def norm(x, name):
        return x / (x.square().mean(-1, keepdim=True) + cfg["rms_norm_eps"]).sqrt() * w[name].double()

    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = norm(x, p + "input_layernorm.weight")
        q, k, v = (_mm(h, w[p + f"self_attn.{n}_proj.weight"]).reshape(len(x), -1, D) for n in "qkv")
        q, k = _rotate(q, pos, freq), _rotate(k, pos, freq)
        x = x + _mm(_each(lens, lambda a, b, c: _attend(a, b, c, D ** -0.5), q, k, v).reshape(len(x), -1), w[p + "self_attn.o_proj.weight"])
        del q, k, v
        h = norm(x, p + "post_attention_layernorm.weight")
        gate, up, down = (w[p + f"mlp.{n}_proj.weight"].double() for n in ("gate", "up", "down"))
        for a in range(0, len(x), 8192):
            b = h[a:a + 8192]
            x[a:a + 8192] += (torch.nn.functional.silu(b @ gate.T) * (b @ up.T)) @ down.T
    head = w["model.embed_tokens.weight"] if cfg["tie_word_embeddings"] else w["lm_head.weight"]
    return norm(x, "model.norm.weight"), head


def _exact_suripel(cfg, w, seqs):
    eps, lens = cfg["norm"]["eps"], [len(t) for t in seqs]
    x = w["embed"][torch.as_tensor(np.concatenate(seqs), device="cuda")].double()
    pos = torch.cat([torch.arange(n, device="cuda") for n in lens])

    def norm(x, name):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], eps=eps) * w[name].double()

    def div(x):
        return x / (x.square().mean(-1, keepdim=True) + eps).sqrt()

    def conv(u, name):
        taps = w[name].double()

        def one(u):
            k = taps.shape[1]
            z = torch.cat([u.new_zeros((k - 1, u.shape[1])), u])
            return sum(z[j:j + len(u)] * taps[:, j] for j in range(k))
        return _each(lens, one, u)

    def recur(q, k, v, decay, beta=None):
        """``S <- decay S + k (v or beta (v - S^T k))^T``, ``o = S^T q`` a token and head; all sequences side by side."""
        starts = np.concatenate([[0], np.cumsum(lens)])
        out = torch.empty((len(q), q.shape[1], v.shape[2]), dtype=q.dtype, device=q.device)
        S = q.new_zeros((len(lens), q.shape[1], q.shape[2], v.shape[2]))
        for t in range(max(lens)):
            live = [i for i, n in enumerate(lens) if t < n]
            rows = torch.as_tensor(starts[live] + t, device="cuda")
            kt, s = k[rows], S[live] * (decay[rows] if decay.dim() == 2 else decay[None])[:, :, None, None]
            u = v[rows] if beta is None else beta[rows][:, :, None] * (v[rows] - (s * kt[..., None]).sum(2))
            s = s + kt[..., None] * u[:, :, None, :]
            S[live] = s
            out[rows] = (s * q[rows][..., None]).sum(2)
        return out

    kvs = {}
    for i, layer in enumerate(cfg["layers"]):
        p, m, kind = f"l{i}.", layer["mixer"], layer["type"]
        H, D, Dv = m["heads"], m["dim"], m["vdim"]
        h = norm(x, p + "norm1")
        h = h + conv(h, p + "canon1")

        def proj(name, heads):
            y = _mm(h, w[p + "mix." + name])
            if "conv" in m:
                y = conv(y, p + "mix." + name + ".conv")
            if kind == "delta":
                y = torch.nn.functional.silu(y)
            return y.reshape(len(x), heads, -1)

        if kind == "attention":
            G = m["kv_heads"]
            q = proj("q", H)
            kvs[i] = kvs[m["kv_from"]] if "kv_from" in m else (proj("k", G), proj("v", G))
            o = _each(lens, lambda a, b, c: _attend(a, b, c, m["scale"], m["mask"]["size"], m["mask"]["pool"]), q, *kvs[i]).reshape(len(x), -1)
        elif kind == "delta":
            G = m["kv_heads"]
            q, k, v = proj("q", G), proj("k", G), proj("v", H)
            q, k = (z / (z.square().sum(-1, keepdim=True) + 1e-6).sqrt() for z in (q, k))
            q, k = (q * D ** -0.5).repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1)
            beta = torch.sigmoid(_mm(h, w[p + "mix.b"]))
            decay = torch.exp(-torch.exp(w[p + "mix.A_log"].double())
                              * torch.nn.functional.softplus(_mm(h, w[p + "mix.a"]) + w[p + "mix.dt_bias"].double()))
            o = div(recur(q, k, v, decay, beta)) * w[p + "mix.norm"].double()
            o = o.reshape(len(x), -1) * torch.nn.functional.silu(_mm(h, w[p + "mix.g"]))
        else:
            q, k, v = proj("q", H), proj("k", H), proj("v", H)
            freq = _inv_freq(m["rot"]["dims"], m["rot"]["base"])
            q, k = _rotate(q, pos, freq), _rotate(k, pos, freq) * D ** -0.5
            o = div(recur(q, k, v, torch.tensor(m["decay"], dtype=torch.float64, device="cuda"))).reshape(len(x), -1)
            o = o * torch.nn.functional.silu(_mm(h, w[p + "mix.g"]))
        x = x + _mm(o, w[p + "mix.o"])
        h = norm(x, p + "norm2")
        h = h + conv(h, p + "canon2")
        a, b, c, e = w[p + "mlp.act"].double()
        for at in range(0, len(x), 8192):
            z = _mm(h[at:at + 8192], w[p + "mlp.up"])
            x[at:at + 8192] += _mm(a * div(z) + b * div(z * z) + c * div(z * z * z) + e, w[p + "mlp.down"])
    return norm(x, "final.norm"), w["head"]


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None
    cfg = MODELS[case["model"]]
    vocab, w = _vocab(cfg), _weights(cfg, case["dtype"], seed)
    run_model = _exact_suripel if cfg.get("architecture") == "Suripel" else _exact_llama
    if kind in ("decode", "mixed"):
        seqs, nxt = _cached(case, seed), _tokens(seed + 3, vocab, ROOM, case["batch"])
        more = 2 if kind == "decode" else 1         # (prepare has run the first decoded token)
        seqs = [np.concatenate([t, nxt[:more, i]]) for i, t in enumerate(seqs)]
        if kind == "mixed":
            seqs.insert(0, _tokens(seed + 5, vocab, case["tokens"]))
        places = [[len(t) - 1 for t in seqs]]
    elif kind == "prompt":
        seqs = [_tokens(seed + 5, vocab, case["tokens"])]
        n = len(seqs[0])
        places = [[list(range(a, min(n, a + PORTION)))] for a in range(0, n, PORTION)] if case["score"] else [[n - 1]]
    else:
        lens, nxt = _replay_lengths(case, seed), _tokens(seed + 3, vocab, case["new"], case["requests"])
        seqs = [np.concatenate([_tokens(seed * 1000 + 17 + i, vocab, n), nxt[:, i]]) for i, n in enumerate(lens)]
        places = [[n - 1 + k for n in lens] for k in range(case["new"] + 1)]
    h, head = run_model(cfg, w, seqs)
    first = np.concatenate([[0], np.cumsum([len(t) for t in seqs])])[:-1]
    got = []
    for at in places:
        rows = np.concatenate([f + np.atleast_1d(p) for f, p in zip(first, at)])
        got.append(_mm(h[torch.as_tensor(rows, device="cuda")], head))
    if kind in ("decode", "mixed"):
        return got[0]
    return got
