"""The work that users of this engine have it do, as cases to time and to compare: prompts, decoded tokens and both in one
step, through `Engine.step` and the sampler, from a tiny 32-bit replay to a mixed step of the 2.1B size.

A case is a dict of plain values:
  kind      "replay" (a few prompts, then given tokens one at a time, all logits), "decode" (one token for each of `batch`
            requests), "prefill" (`prompts` prompts in one step) or "mixed" (decoded tokens beside a portion of a prompt)
  model     a named size ("tiny", "0.9B", "2.1B"), or a design ("Tikalix", "Fesupel", "Fikevik") of 4 layers of `width`
Random weights, uniform token ids; tokens to decode are given (as a replay gives them), so that one close arg-max does not
change everything after it.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from tiny_inference_server_amd.__main__ import size_config
from tiny_inference_server_amd.config import ARCHITECTURES, config_from_dict
from tiny_inference_server_amd.engine import Engine
from tiny_inference_server_amd.sampling.params import SamplingParams
from tiny_inference_server_amd.sampling.sampler import Sampler
from tiny_inference_server_amd.weights.loader import spec_tensors

DEV = "cuda:0"
PAGE = 16
PORTION = 2048        # tokens of a prompt in one step
ROOM = 1024           # tokens a decoding request may take before its context is fed again
VOCAB = 32000         # of the designs
MOE_EXPERTS, MOE_TOP = 8, 2
# the reference's sampling options
SAMPLING = dict(temperature=0.9, top_k=50, top_p=0.95, rep_penalty=1.1)


# ---- the cases --------------------------------------------------------------------------------------------------------

def listed():
    return [
        # the smallest calls there are: logits of a small 32-bit model, checked against another implementation
        dict(name="tiny_replay", kind="replay", model="tiny", prompts=3, longest=33, tokens=16),
        # one user's chat at the headline size: latency of a token
        dict(name="decode_1", kind="decode", model="0.9B", batch=1, context=900, spread=0.0, sample=False),
        # the headline: batch 8 near 4,096 tokens
        dict(name="decode_8", kind="decode", model="0.9B", batch=8, context=4000, spread=0.02, sample=False),
        # a full server: 64 requests of very different lengths, sampled with the reference's options
        dict(name="decode_64_sampled", kind="decode", model="0.9B", batch=64, context=4096, spread=0.94, sample=True),
        # the headline's prompt
        dict(name="prefill_2048", kind="prefill", model="0.9B", prompts=1, longest=2048, spread=0.0, heads=False, score=False),
        # several users' prompts of odd lengths in one step, with the prediction heads' logits
        dict(name="prefill_ragged", kind="prefill", model="0.9B", prompts=6, longest=611, spread=0.95, heads=True, score=False),
        # serving under load: decoded tokens beside a portion of a new prompt
        dict(name="mixed_2.1B", kind="mixed", model="2.1B", batch=32, context=4096, spread=0.9, portion=1500),
        # the further designs: attention and a mixture of experts
        dict(name="tikalix_prefill", kind="prefill", model="Tikalix", width=2048, prompts=1, longest=2048, spread=0.0, heads=False, score=False),
        dict(name="tikalix_decode", kind="decode", model="Tikalix", width=2048, batch=8, context=2000, spread=0.5, sample=False),
        # attention with mixed weights beside a delta rule, and experts in groups
        dict(name="fesupel_prefill", kind="prefill", model="Fesupel", width=2048, prompts=1, longest=1531, spread=0.0, heads=False, score=False),
        dict(name="fesupel_decode", kind="decode", model="Fesupel", width=1024, batch=5, context=700, spread=0.5, sample=False),
        # windowed attention beside a matrix memory, gated linear attention; a text is scored: logits of every position
        dict(name="fikevik_score", kind="prefill", model="Fikevik", width=2048, prompts=2, longest=1200, spread=0.5, heads=False, score=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["replay", "decode", "decode", "decode", "prefill", "prefill", "prefill", "mixed"])
    if kind == "replay":
        return dict(kind=kind, model="tiny", prompts=rng.randint(1, 4), longest=rng.randint(6, 100), tokens=rng.randint(4, 32))
    spread = round(rng.choice([0.0, rng.uniform(0.05, 0.95)]), 3)
    if kind == "mixed":
        batch = _log_int(rng, 4, 32)
        return dict(kind=kind, model=rng.choice(["0.9B", "2.1B"]), batch=batch, context=_log_int(rng, 300, 4096),
                    spread=max(spread, 0.5), portion=_log_int(rng, 100, 1500))
    model = rng.choice(["0.9B", "0.9B", "Tikalix", "Fesupel", "Fikevik"])
    case = dict(kind=kind, model=model, spread=spread)
    if model != "0.9B":
        case["width"] = rng.choice([1024, 2048])
    if kind == "decode":
        case["batch"] = _log_int(rng, 1, 64 if model == "0.9B" else 32)
        most = 4096 if case["batch"] <= 16 else 2100
        case["context"] = _log_int(rng, 40, most if model == "0.9B" else 2048)
        case["sample"] = rng.random() < 0.4
        return case
    case["prompts"] = rng.choice([1, 1, rng.randint(2, 8)])
    case["longest"] = _log_int(rng, 40, 4096 // case["prompts"] if model == "0.9B" else 2048 // case["prompts"])
    case["heads"] = model == "0.9B" and rng.random() < 0.3
    case["score"] = model != "0.9B" and rng.random() < 0.4
    return case


# ---- models and inputs ------------------------------------------------------------------------------------------------

def _design(case):
    """The configuration of a design, as a config.json holds it: 4 layers, heads of 128 channels, the feed-forward 2.75 times
    the width; a mixture has 8 experts of which a token takes 2."""
    name, width = case["model"], case["width"]
    heads, kv, ff = width // 128, width // 512, 11 * width // 4
    moe = {"kind": "moe", "expert": {"ff": ff // MOE_TOP, "limit": 7.0}, "router": {"experts": MOE_EXPERTS, "top": MOE_TOP},
           "shared": {"ff": ff // 4, "limit": 7.0}}
    raw = {"architecture": name, "vocab": VOCAB, "width": width, "norm": {"eps": 1e-5}}
    if name == "Tikalix":
        mixer = {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "softcap": 30.0,
                 "rot": {"dims": 128, "base": 500000.0, "scaling": {"factor": 4.0, "original": 8192, "fast": 32.0, "slow": 1.0}}}
        raw.update(embedding={"scale": width ** 0.5}, residual_mult=0.5,
                   layers=[{"type": "attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": ff} if i % 2 == 0 else moe} for i in range(4)])
    elif name == "Fesupel":
        moe["router"].update(identity=1, groups={"count": 3, "keep": 2})
        mixer = {"left": {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "softcap": 30.0, "mask": {"size": 1024},
                          "rot": {"dims": 64, "base": 1000000.0, "scaling": {"factor": 4.0, "low": 1.0, "high": 4.0, "original": 8192}}},
                 "right": {"heads": heads // 2, "kv_heads": max(1, kv // 2), "dim": 128, "vdim": 256, "conv": 4, "decay_rank": 64, "gate_rank": 64}}
        raw.update(embedding={"scale": width ** 0.5}, token_side={"dim": 64},
                   layers=[{"type": "parallel", "mixer": mixer, "mlp": {"kind": "dense", "ff": ff} if i % 2 == 0 else moe} for i in range(4)])
    else:
        dense = {"kind": "dense", "ff": ff}
        par = {"type": "parallel", "mlp": dense,
               "mixer": {"left": {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "mask": {"size": 1024},
                                  "rot": {"dims": 64, "base": 1000000.0}, "scale": 128 ** -0.5},
                         "right": {"heads": heads // 2, "dim": 128, "vdim": 256, "gate_cap": 12.0}, "left_scale": 1.0, "right_scale": 1.0}}
        gla = {"type": "gla", "mlp": dense, "mixer": {"heads": heads // 2, "dim": 128, "vdim": 256, "tau": 8.0, "rank": 32}}
        raw.update(embedding={"scale": 1.0}, postln_alpha=1.0, layers=[par if i % 2 == 0 else gla for i in range(4)])
    return raw


def _config(case):
    return config_from_dict(_design(case)) if "width" in case else size_config(case["model"])


def _dtype(case):
    return "float32" if case["kind"] == "replay" else "bfloat16"


def _shapes(case):
    cfg = _config(case)
    return spec_tensors(ARCHITECTURES.get(cfg.architecture).build_spec(cfg))


def _tensors(case, seed):
    """Random weights by name, N(0, 0.02) with gains of 1 as the repository's own random models have them; what a trained model
    of a design has at another size (gates, decays, taps, biases, the scale around which a gain is stored) is drawn at that
    size, and a token has two experts it prefers, as trained routers do: with random ones every second comparison is a tie."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1000 + seed)
    dtype = getattr(torch, _dtype(case))

    def normal(shape, std):
        return torch.randn(shape, generator=gen, device=DEV) * std

    def uniform(shape, lo, hi):
        return torch.rand(shape, generator=gen, device=DEV) * (hi - lo) + lo

    out = {}
    for name, shape in sorted(_shapes(case).items()):
        last = name.rsplit(".", 1)[-1]
        if len(shape) == 2:
            t = uniform(shape, -0.5, 0.5) if last == "conv" else normal(shape, 0.02)
            if last == "talk":
                t = t + torch.eye(shape[0], device=DEV)
        elif last == "b":
            t = normal(shape, 0.02) + (4.0 if name.endswith((".f.b", ".a2.b")) else 0.0)
        elif last == "A_log":
            t = torch.log(uniform(shape, 1.0, 16.0))
        elif last == "dt_bias":
            t = torch.log(torch.expm1(uniform(shape, 0.001, 0.1)))
        elif last == "pb":
            t = normal(shape, 0.1) - math.log(512.0)
        elif last == "correction":
            t = normal(shape, 0.01)
        elif case["model"] == "Tikalix" and "norm" in last:
            t = normal(shape, 0.05)
        else:
            t = torch.ones(shape, device=DEV)
        out[name] = t
    routers = sorted(n for n in out if n.endswith(".router"))
    if routers:
        n = out[routers[0]].shape[0]
        first = torch.randint(0, n, (VOCAB,), generator=gen, device=DEV)
        second = (first + torch.randint(1, n, (VOCAB,), generator=gen, device=DEV)) % n
        much = 0.6 if case["model"] == "Fesupel" else 0.2
        for r in routers:
            unit = out[r] / out[r].norm(dim=1, keepdim=True)
            out["embed"] += much * (unit[first] + 0.8 * unit[second])
    return {n: t.to(dtype) for n, t in out.items()}


def _lengths(case, n, longest, rng):
    """`n` lengths up to `longest`, spread evenly over the last `spread` of it, in any order; one has the full length."""
    lens = [max(4, int(round(longest * (1.0 - case.get("spread", 0.9) * i / max(1, n - 1))))) for i in range(n)]
    return [lens[i] for i in rng.permutation(n)]


def _sequences(case, seed):
    """(prompts or contexts, tokens to decode per request): lists of token ids."""
    rng = np.random.RandomState(seed % (1 << 31))
    vocab = VOCAB if "width" in case else _config(case).vocab_size
    n = case.get("batch", case.get("prompts"))
    longest = case.get("context", case.get("longest"))
    lens = _lengths(case, n, longest, rng)
    if case["kind"] == "replay":
        lens[0] = min(lens[0], 5)
    texts = [rng.randint(0, vocab, k).tolist() for k in lens]
    given = rng.randint(0, vocab, (ROOM, n)).tolist()
    portion = rng.randint(0, vocab, case["portion"]).tolist() if "portion" in case else None
    return texts, given, portion


def _feed(state):
    """The contexts of the decoding requests, in portions."""
    engine = state["engine"]
    for rid, text in enumerate(state["texts"]):
        if rid in engine.requests:
            engine.close(rid)
        for p in range(0, len(text), PORTION):
            engine.step([(rid, text[p:p + PORTION], [])])
    state["at"] = 0


def prepare(case, seed):
    texts, given, portion = _sequences(case, seed)
    kind = case["kind"]
    grows = ROOM if kind in ("decode", "mixed") else case.get("tokens", 0)
    pool = sum(-(-(len(t) + grows) // PAGE) * PAGE for t in texts) + (case.get("portion", 0) + PAGE)
    engine = Engine(config=_config(case), tensors=_tensors(case, seed), dtype=_dtype(case), page_size=PAGE, max_tokens=pool,
                    max_requests=len(texts) + 1, device=DEV)
    state = dict(case=case, engine=engine, texts=texts, given=given, portion=portion, at=0, sampler=None)
    if kind in ("decode", "mixed"):
        _feed(state)
        if case.get("sample"):
            state["sampler"] = Sampler(engine.ops, engine.spec.vocab_size, engine.max_requests)
            state["params"] = [SamplingParams(seed=seed + i, **SAMPLING) for i in range(len(texts))]
    return state


# ---- one pass ---------------------------------------------------------------------------------------------------------

def _pick(state, logits):
    """The tokens that a program reads back after a step: arg-max, or sampled with the request's options. (Few tokens are read
    back and not compared: a single close call, which its logits show to be one, would be a difference of the whole.)"""
    if state["sampler"] is None:
        tokens = np.asarray(state["engine"].ops.argmax(logits).tolist())
        return tokens if len(tokens) >= 4 else None
    n = len(state["texts"])
    slots = [state["engine"].requests[r][0] for r in range(n)]
    tokens = np.asarray(state["sampler"].sample(logits, state["params"], [state["at"]] * n, state["texts"], slots, list(range(n))))
    return tokens if n >= 4 else None


def run(state):
    case, engine = state["case"], state["engine"]
    return {"replay": _run_replay, "decode": _run_decode, "prefill": _run_prefill, "mixed": _run_mixed}[case["kind"]](state, case, engine)


def _run_replay(state, case, engine):
    texts = state["texts"]
    n = len(texts)
    out = engine.step([(r, t, [len(t) - 1]) for r, t in enumerate(texts)], heads=True)
    logits, heads = [out.logits], list(out.head_logits)
    for k in range(case["tokens"]):
        # (a captured step's logits are valid until the next step)
        logits.append(engine.step([(r, [state["given"][k][r]], [0]) for r in range(n)]).logits.clone())
    for r in range(n):
        engine.close(r)
    return {"logits": torch.stack(logits), "heads": heads}


def _run_decode(state, case, engine):
    if state["at"] == ROOM:
        _feed(state)
    given = state["given"][state["at"]]
    out = engine.step([(r, [t], [0]) for r, t in enumerate(given)])
    tokens = _pick(state, out.logits)
    state["at"] += 1
    return {"logits": out.logits, "tokens": tokens}


def _run_prefill(state, case, engine):
    texts = state["texts"]
    out = engine.step([(r, t, range(len(t)) if case["score"] else [len(t) - 1]) for r, t in enumerate(texts)], heads=case["heads"])
    result = {"logits": out.logits, "heads": out.head_logits}
    if not case["score"]:
        result["tokens"] = _pick(state, out.logits)
    for r in range(len(texts)):
        engine.close(r)
    return result


def _run_mixed(state, case, engine):
    if state["at"] == ROOM:
        _feed(state)
    given, portion = state["given"][state["at"]], state["portion"]
    out = engine.step([(r, [t], [0]) for r, t in enumerate(given)] + [("new", portion, [len(portion) - 1])])
    tokens = np.asarray(engine.ops.argmax(out.logits).tolist())
    state["at"] += 1
    engine.close("new")
    return {"logits": out.logits, "tokens": tokens}


# ---- what a pass cannot do without ------------------------------------------------------------------------------------

def work(case):
    """Every matrix once (of a mixture's experts as many as there are choices, at most all), the keys and values or states of
    the requests once, the logits; two operations a matrix element and token, four a (token, key) pair and channel."""
    texts, _, portion = _sequences(case, 0)
    shapes = _shapes(case)
    elem = 4 if _dtype(case) == "float32" else 2
    table = {"embed", "embedding.weight", "side.embed"}
    tied = "head" not in shapes and "lm_head.weight" not in shapes
    expert = sum(s[0] * s[1] for n, s in shapes.items() if len(s) == 2 and ".mlp.e" in n)
    dense = sum(s[0] * s[1] for n, s in shapes.items() if len(s) == 2 and ".mlp.e" not in n and n not in table
                and n not in ("head", "lm_head.weight"))
    cfg = _config(case)
    if "width" in case:
        width, vocab, layers = case["width"], VOCAB, 4
        kv_channels, channels = width // 4, width
    else:
        width, vocab, layers = cfg.d_model, cfg.vocab_size, cfg.n_layers + cfg.mtp_heads
        kv_channels, channels = width // cfg.group_size, width
    out_table = width * vocab

    def step(rows, wanted, keys, pairs):
        read = dense + min(1.0, rows * MOE_TOP / MOE_EXPERTS) * expert + out_table
        moved = read * elem + keys * layers * 2 * kv_channels * elem + rows * (width + layers * 2 * kv_channels) * elem + wanted * vocab * 4
        return moved, 2.0 * rows * (dense + expert * MOE_TOP / MOE_EXPERTS) + 2.0 * wanted * out_table + 4.0 * pairs * channels * layers

    assert tied == ("width" not in case)
    kind, n = case["kind"], len(texts)
    window = {"Fikevik": 1024, "Fesupel": 1024}.get(case["model"], 1 << 30)
    reach = lambda k: min(k, window)  # noqa: E731
    causal = lambda k: sum(reach(i + 1) for i in range(k))  # noqa: E731
    steps = []
    if kind in ("replay", "prefill"):
        rows = sum(len(t) for t in texts)
        wanted = (rows if case.get("score") else n) * (1 + (cfg.mtp_heads if case.get("heads") or kind == "replay" else 0))
        steps.append(step(rows, wanted, 0, sum(causal(len(t)) for t in texts)))
        for k in range(case.get("tokens", 0)):
            keys = sum(len(t) + k + 1 for t in texts)
            steps.append(step(n, n, keys, keys))
    else:
        keys = sum(reach(len(t) + 1) for t in texts)
        p = len(portion) if portion else 0
        steps.append(step(n + p, n + (1 if p else 0), keys, keys + causal(p)))
    return {"bytes": float(sum(s[0] for s in steps)), "flops": float(sum(s[1] for s in steps))}


def tolerance(case):
    """About four times what the engine's outputs lie off the 64-bit ones: 2.7e-7 in 32 bits; in bf16 0.018 through the 0.9B
    size's 30 layers, 0.033 through the 2.1B size's 40, 0.003 to 0.007 through a design's 4. The largest of a row's
    thousands of differences is some five times their root mean square. Tokens: close calls of the arg-max or the draw."""
    if case["kind"] == "replay":
        return {"rel": 1.2e-6, "max": 1e-5}
    rel = 0.025 if "width" in case else 0.13 if case["model"] == "2.1B" else 0.07
    n = case.get("batch", case.get("prompts"))
    return {"rel": rel, "max": 5 * rel, "differ": 0.5 if n < 8 else 0.3}


# ---- the same in 64 bits, without this repository's kernels and cache -------------------------------------------------

F64 = torch.float64


def exact(case, seed):
    texts, given, portion = _sequences(case, seed)
    raw = _tensors(case, seed)
    w = {n: t.to(F64) for n, t in raw.items()}
    del raw
    if "width" in case:
        design = _design(case)
        full = {"Tikalix": _tikalix, "Fesupel": _fesupel, "Fikevik": _fikevik}[case["model"]]
        forward = lambda ids: (full(design, w, ids), [])  # noqa: E731
        table, lags = w["head"], []
    else:
        cfg = _config(case)
        forward = lambda ids: _gqa(cfg, w, ids, heads=case.get("heads") or case["kind"] == "replay")  # noqa: E731
        table, lags = w["lm_head.weight"] if "lm_head.weight" in w else w["embedding.weight"], list(range(1, cfg.mtp_heads + 1))
    kind = case["kind"]
    if kind == "replay":
        outs = [forward(t + [given[k][r] for k in range(case["tokens"])]) for r, t in enumerate(texts)]
        last = [len(t) - 1 for t in texts]
        rows = torch.stack([torch.stack([o[0][p + k] for o, p in zip(outs, last)]) for k in range(case["tokens"] + 1)])
        return {"logits": rows @ table.T, "heads": [torch.stack([o[1][j - 1][p - j] for o, p in zip(outs, last)]) @ table.T for j in lags]}
    if kind == "prefill":
        outs = [forward(t) for t in texts]
        if case["score"]:
            return {"logits": torch.cat([o[0] for o in outs]) @ table.T, "heads": None}
        last = [len(t) - 1 for t in texts]
        heads = [torch.stack([o[1][j - 1][p - j] for o, p in zip(outs, last)]) @ table.T for j in lags] if case["heads"] else None
        return {"logits": torch.stack([o[0][p] for o, p in zip(outs, last)]) @ table.T, "heads": heads, "tokens": None}
    rows = [forward(t + [given[0][r]])[0][-1] for r, t in enumerate(texts)]
    if portion:
        rows.append(forward(portion)[0][-1])
    return {"logits": torch.stack(rows) @ table.T, "tokens": None}


def _attend(q, k, v, scale, weights):
    """q [T, H, D], k [T, G, D], v [T, G, V]; weights(scores [H / G, rows, T], first row) -> the same shape."""
    T, H, D = q.shape
    G = k.shape[1]
    out = q.new_empty(T, H, v.shape[2])
    for g in range(G):
        for a in range(0, T, 1024):
            qs = q[a:a + 1024, g * (H // G):(g + 1) * (H // G)].transpose(0, 1).contiguous()
            end = min(T, a + 1024)
            p = weights(qs @ k[:end, g].T.contiguous() * scale, a)
            out[a:a + 1024, g * (H // G):(g + 1) * (H // G)] = (p @ v[:end, g].contiguous()).transpose(0, 1)
    return out


def _seen(s, first, window=0, chunk=0):
    i = torch.arange(first, first + s.shape[-2], device=s.device)[:, None]
    j = torch.arange(s.shape[-1], device=s.device)[None]
    ok = j <= i
    if window:
        ok = ok & (j > i - window)
    if chunk:
        ok = ok & (i // chunk == j // chunk)
    return ok


def _softmax(window=0, cap=0.0):
    def weights(s, first):
        if cap:
            s = cap * torch.tanh(s / cap)
        return torch.softmax(s.masked_fill(~_seen(s, first, window), -math.inf), dim=-1)
    return weights


def _rotate(x, freqs, dims, factor=1.0, pairs=False):
    """Channels i and i + dims / 2 (or 2 i and 2 i + 1 with `pairs`) turn by position * freqs[i]; channels from dims on stay."""
    ang = torch.arange(x.shape[0], device=x.device, dtype=F64)[:, None, None] * torch.as_tensor(freqs, dtype=F64, device=x.device)
    c, s = torch.cos(ang) * factor, torch.sin(ang) * factor
    y = x.clone()
    u, v = (slice(0, dims, 2), slice(1, dims, 2)) if pairs else (slice(0, dims // 2), slice(dims // 2, dims))
    y[..., u], y[..., v] = x[..., u] * c - x[..., v] * s, x[..., v] * c + x[..., u] * s
    return y


def _unit(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _gqa(cfg, w, ids, heads):
    """Rows after the closing norm: of the trunk, and (asked for) of every prediction head."""
    H, G, D = cfg.n_heads, cfg.n_heads // cfg.group_size, cfg.d_model // cfg.n_heads
    freqs = [cfg.rope_base ** (-2.0 * i / D) for i in range(D // 2)]

    def norm(x, gain):
        return x * math.sqrt(x.shape[-1]) / (x.norm(dim=-1, keepdim=True) + cfg.rms_eps) * gain

    def block(x, p):
        T = x.shape[0]
        a = norm(x, w[p + "att.rms_norm_att.scale"])
        q = (a @ w[p + "att.q_proj.weight"]).view(T, H, D)
        k, v = (a @ w[p + "att.kv_proj.weight"]).view(T, 2, G, D).unbind(1)
        o = _attend(_rotate(q, freqs, D), _rotate(k, freqs, D), v, D ** -0.5, _softmax())
        x = x + o.reshape(T, -1) @ w[p + "att.linear_proj.weight"]
        f = norm(x, w[p + "rms_norm_ffn.scale"])
        return x + (_silu(f @ w[p + "ffn.swig.linear1.weight"]) * (f @ w[p + "ffn.swig.linear2.weight"])) @ w[p + "ffn.fc.weight"]

    tokens = torch.tensor(ids, device=DEV)
    x = w["embedding.weight"][tokens]
    for i in range(cfg.n_layers):
        x = block(x, f"transformer_block_list.{i}.")
    stages = [norm(x, w["rms_out.scale"])]
    for i in range(cfg.mtp_heads if heads else 0):
        p, n = f"mtp_heads_list.{i}.", len(ids) - 1 - i
        e = norm(w["embedding.weight"][tokens[1 + i:]], w[p + "rms_embed.scale"])
        stages.append(norm(block(torch.cat([stages[-1][:n], e], -1) @ w[p + "proj.weight"], p + "trans_block."), w[p + "rms_out.scale"]))
    return stages[0], stages[1:]


def _expert(h, w, p, limit):
    g = torch.clamp(h @ w[p + "gate"].T, max=limit)
    u = torch.clamp(h @ w[p + "up"].T, -limit, limit)
    return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w[p + "down"].T


def _mixture(h, w, p, mlp, ids, share):
    y = torch.zeros_like(h)
    E = mlp["router"]["experts"]
    for e in range(E + mlp["router"].get("identity", 0)):
        part = (share * (ids == e)).sum(-1, keepdim=True)
        rows = part[:, 0] != 0
        y[rows] += part[rows] * (_expert(h[rows], w, f"{p}e{e}.", mlp["expert"]["limit"]) if e < E else h[rows])
    return y


def _feed_forward(h, w, p, mlp):
    """A squared relu, or a mixture beside a shared expert: chosen and weighed by a softmax (Tikalix: over the chosen scores;
    with groups: chosen with a correction among the best groups, weights the plain scores over their sum)."""
    if mlp["kind"] == "dense":
        return torch.relu(h @ w[p + "up"].T) ** 2 @ w[p + "down"].T
    r, z = mlp["router"], h @ w[p + "router"].T
    shared = _expert(h, w, p + "shared.", mlp["shared"]["limit"])
    if "groups" not in r:
        best = torch.topk(z, r["top"], dim=-1)
        return _mixture(h, w, p, mlp, best.indices, torch.softmax(best.values, -1)) + shared
    scores = torch.softmax(z, -1)
    c = scores + w[p + "correction"]
    T, count = c.shape[0], r["groups"]["count"]
    top_groups = torch.topk(c.view(T, count, -1).amax(-1), r["groups"]["keep"], dim=-1).indices
    keep = torch.zeros(T, count, dtype=torch.bool, device=c.device).scatter_(1, top_groups, True)
    c = c.masked_fill(~keep.repeat_interleave(c.shape[1] // count, 1), -math.inf)
    ids = torch.topk(c, r["top"], dim=-1).indices
    s = torch.gather(scores, 1, ids)
    return _mixture(h, w, p, mlp, ids, s / (s.sum(-1, keepdim=True) + 1e-20)) + shared * torch.sigmoid(h @ w[p + "shared.sg"].T)


def _tikalix(cfg, w, ids):
    eps, mult = cfg["norm"]["eps"], cfg["residual_mult"]
    x = w["embed"][torch.tensor(ids, device=DEV)] * cfg["embedding"]["scale"]
    T = x.shape[0]
    for i, entry in enumerate(cfg["layers"]):
        p, m, sc = f"l{i}.", entry["mixer"], entry["mixer"]["rot"]["scaling"]
        H, G, D, V, dims, base = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["rot"]["dims"], m["rot"]["base"]
        at = lambda turns: dims * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), dims - 1)
        freqs = []
        for j in range(dims // 2):
            f, r = base ** (-2.0 * j / dims), min(max((j - lo) / max(hi - lo, 0.001), 0.0), 1.0)
            freqs.append(f / sc["factor"] * r + f * (1.0 - r))
        turn = lambda t: _unit(_rotate(t, freqs, dims, 0.1 * math.log(sc["factor"]) + 1.0), eps)  # noqa: E731
        q = (x @ w[p + "mix.q"].T + w[p + "mix.q.b"]).view(T, H, D)
        k = (x @ w[p + "mix.k"].T + w[p + "mix.k.b"]).view(T, G, D)
        v = (x @ w[p + "mix.v"].T + w[p + "mix.v.b"]).view(T, G, V)
        o = _attend(turn(q), turn(k), v, m["scale"], _softmax(cap=m["softcap"])).reshape(T, -1)
        x = x + mult * _unit((o * torch.sigmoid(x @ w[p + "mix.g"].T)) @ w[p + "mix.o"].T, eps) * (1.0 + w[p + "norm1"])
        x = x + mult * _unit(_feed_forward(x, w, p + "mlp.", entry["mlp"]), eps) * (1.0 + w[p + "norm2"])
    return _unit(x, eps) * (1.0 + w["final.norm"])


def _conv(x, taps):
    """Causal, per channel: the last tap meets the row itself."""
    K = taps.shape[1]
    padded = torch.cat([x.new_zeros(K - 1, x.shape[1]), x])
    return sum(padded[j:j + x.shape[0]] * taps[:, j] for j in range(K))


def _fesupel(cfg, w, ids):
    eps = cfg["norm"]["eps"]
    tokens = torch.tensor(ids, device=DEV)
    x = w["embed"][tokens] * cfg["embedding"]["scale"]
    T = x.shape[0]
    normed = lambda t, gain: _unit(t, eps) * gain  # noqa: E731
    for i, entry in enumerate(cfg["layers"]):
        p, m = f"l{i}.", entry["mixer"]["left"]
        h = normed(x, w[p + "norm1"])
        H, G, D, V, dims, sc = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["rot"]["dims"], m["rot"]["scaling"]
        freqs = []
        for j in range(dims // 2):
            f = m["rot"]["base"] ** (-2.0 * j / dims)
            r = min(max((sc["original"] * f / (2.0 * math.pi) - sc["low"]) / (sc["high"] - sc["low"]), 0.0), 1.0)
            freqs.append((1.0 - r) * f / sc["factor"] + r * f)
        l = p + "mix.left."
        q = _rotate((h @ w[l + "q"].T + w[l + "q.b"]).view(T, H, D), freqs, dims)
        k = _rotate((h @ w[l + "k"].T + w[l + "k.b"]).view(T, G, D), freqs, dims)
        v = (h @ w[l + "v"].T + w[l + "v.b"]).view(T, G, V)
        left = x.new_zeros(T, H, V)
        size = m["mask"]["size"]
        for a in range(0, T, size):          # a chunk of positions at a time; every head's weights are a mix of all heads'
            b = min(T, a + size)
            s = torch.stack([q[a:b, n] @ k[a:b, n // (H // G)].T for n in range(H)]) * m["scale"]
            s = torch.sigmoid(m["softcap"] * torch.tanh(s / m["softcap"]) + w[l + "pb"][:, None, None]) * _seen(s, 0)
            s = (w[l + "talk"] @ s.view(H, -1)).view(H, b - a, b - a)
            for n in range(H):
                left[a:b, n] = s[n] @ v[a:b, n // (H // G)]
        left = left.reshape(T, -1) @ w[l + "o"].T
        m, r = entry["mixer"]["right"], p + "mix.right."
        H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k = (_silu(_conv(h @ w[r + n].T, w[r + n + ".conv"])).view(T, G, D).repeat_interleave(H // G, 1) for n in "qk")
        v = _silu(_conv(h @ w[r + "v"].T, w[r + "v.conv"])).view(T, H, V)
        q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        q = q * D ** -0.5
        beta = torch.sigmoid(h @ w[r + "b"].T)
        step = torch.nn.functional.softplus((h @ w[r + "a1"].T) @ w[r + "a2"].T + w[r + "dt_bias"]).view(T, H, D)
        decay = torch.exp(-torch.exp(w[r + "A_log"]).view(1, H, 1) * step)
        S, o = x.new_zeros(H, D, V), x.new_empty(T, H, V)
        for t in range(T):
            S = S * decay[t, :, :, None]
            u = beta[t, :, None, None] * (v[t, :, None] - k[t, :, None] @ S)
            S = torch.baddbmm(S, k[t, :, :, None], u)
            o[t] = (q[t, :, None] @ S)[:, 0]
        gate = torch.sigmoid((h @ w[r + "g1"].T) @ w[r + "g2"].T).view(T, H, V)
        right = (normed(o, w[r + "norm"]) * gate).reshape(T, -1) @ w[r + "o"].T
        y = 0.5 * (normed(left, w[l + "out"]) + normed(right, w[r + "out"]))
        x = x + normed(y, w[p + "norm1b"])
        x = x + normed(_feed_forward(normed(x, w[p + "norm2"]), w, p + "mlp.", entry["mlp"]), w[p + "norm2b"])
        dim = cfg["token_side"]["dim"]
        g = torch.nn.functional.gelu(x @ w[p + "side.gate"].T, approximate="tanh")
        x = x + normed((g * w["side.embed"][tokens][:, i * dim:(i + 1) * dim]) @ w[p + "side.proj"].T, w[p + "side.norm"])
    return normed(x, w["final.norm"])


def _fikevik(cfg, w, ids):
    eps, alpha = cfg["norm"]["eps"], cfg["postln_alpha"]
    x = w["embed"][torch.tensor(ids, device=DEV)] * cfg["embedding"]["scale"]
    T = x.shape[0]
    for i, entry in enumerate(cfg["layers"]):
        p, m = f"l{i}.", entry["mixer"]
        r = m["right"] if entry["type"] == "parallel" else m
        pre = p + "mix.right." if entry["type"] == "parallel" else p + "mix."
        H, D, V = r["heads"], r["dim"], r["vdim"]
        q = (x @ w[pre + "q"].T).view(T, H, D) * D ** -0.5
        k, v = (x @ w[pre + "k"].T).view(T, H, D), (x @ w[pre + "v"].T).view(T, H, V)
        S, o = x.new_zeros(H, D, V), x.new_empty(T, H, V)
        gate = x @ w[pre + "g"].T
        if entry["type"] == "parallel":
            cap = r["gate_cap"]
            gi = cap * torch.tanh((x @ w[pre + "i"].T + w[pre + "i.b"]) / cap)
            gf = torch.nn.functional.logsigmoid(cap * torch.tanh((x @ w[pre + "f"].T + w[pre + "f.b"]) / cap))
            n, top = x.new_zeros(H, D), x.new_zeros(H)
            for t in range(T):
                new = torch.maximum(gf[t] + top, gi[t])
                keep, take = torch.exp(gf[t] + top - new), torch.exp(gi[t] - new)
                kt = take[:, None] * k[t]
                S = torch.baddbmm(keep[:, None, None] * S, kt[:, :, None], v[t][:, None])
                n, top = keep[:, None] * n + kt, new
                den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
                o[t] = (q[t][:, None] @ S)[:, 0] / den[:, None]
            y = (_unit(o, eps).reshape(T, -1) * w[pre + "norm"] * torch.sigmoid(gate)) @ w[pre + "o"].T
            m, l = m["left"], p + "mix.left."
            H, G, D, V, dims = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["rot"]["dims"]
            freqs = [m["rot"]["base"] ** (-2.0 * j / dims) for j in range(dims // 2)]
            turn = lambda t, gain: _rotate(_unit(t, eps) * gain, freqs, dims, pairs=True)  # noqa: E731
            q = turn((x @ w[l + "q"].T).view(T, H, D), w[l + "q.norm"]) * w[l + "temp"][:, None]
            k = turn((x @ w[l + "k"].T).view(T, G, D), w[l + "k.norm"])
            v = _unit((x @ w[l + "v"].T).view(T, G, V), eps)
            left = _attend(q, k, v, m["scale"], _softmax(window=m["mask"]["size"])).reshape(T, -1) @ w[l + "o"].T
            y = entry["mixer"]["left_scale"] * left + entry["mixer"]["right_scale"] * y
        else:
            z = (x @ w[pre + "a1"].T) @ w[pre + "a2"].T + w[pre + "a2.b"]
            decay = torch.exp(torch.nn.functional.logsigmoid(z) / r["tau"]).view(T, H, D)
            for t in range(T):
                S = torch.baddbmm(decay[t, :, :, None] * S, k[t][:, :, None], v[t][:, None])
                o[t] = (q[t][:, None] @ S)[:, 0]
            y = ((_unit(o, eps) * w[pre + "norm"]).reshape(T, -1) * _silu(gate)) @ w[pre + "o"].T
        x = _unit(alpha * x + y * torch.sigmoid(x @ w[p + "rg1"].T + w[p + "rg1.b"]), eps) * w[p + "norm1"]
        y = (_silu(x @ w[p + "mlp.gate"].T) * (x @ w[p + "mlp.up"].T)) @ w[p + "mlp.down"].T
        x = _unit(alpha * x + y * torch.sigmoid(x @ w[p + "rg2"].T + w[p + "rg2.b"]), eps) * w[p + "norm2"]
    return _unit(x, eps) * w["final.norm"]
