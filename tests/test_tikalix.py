"""The Tikalix architecture on the host: its configuration and spec, the plain implementation's mechanisms against closed
forms, and the engine (step function, cache manager, scheduler, generate) on the torch stand-ins for the kernels against the
plain implementation, in 32-bit."""
import copy
import math
from types import SimpleNamespace

import pytest
import torch

import helpers as H
import plain_tikalix as pt
import tikalix_models as TM
from torch_ops import TorchOps
from tiny_inference_server_amd.config import ARCHITECTURES, ConfigError, config_from_dict, load_config
from tiny_inference_server_amd.engine import Engine
from tiny_inference_server_amd.engine.generate import generate
from tiny_inference_server_amd.ops.hip_ops import HipOps
from tiny_inference_server_amd.parts.attention import slowed_frequencies
from tiny_inference_server_amd.weights.loader import spec_tensors

TOL32 = TM.TOL["float32"]
# the configuration of ones divides single numbers by their own size: where such a number is small, 32-bit rounding is a
# larger share of it
TOL_OF = {"D": 3e-4}
F64 = torch.float64


def model(name, seed=5):
    cfg = TM.CONFIGS[name]
    w = TM.random_weights(cfg, seed)
    return cfg, w, TM.as_f64(w)


def engine_for(cfg, w, **kw):
    kw.setdefault("max_requests", 4)
    kw.setdefault("page_size", 8)
    kw.setdefault("max_tokens", 640)
    return Engine(config=config_from_dict(cfg), tensors={n: t.float() for n, t in w.items()}, dtype="float32",
                  ops=TorchOps(graphs=kw.pop("graphs", False)), **kw)


# ---- configuration and spec ------------------------------------------------------------------------------------

def test_spec_names_every_tensor(tmp_path):
    for name, cfg in TM.CONFIGS.items():
        w = TM.random_weights(cfg, 1)
        c = load_config(TM.write_folder(str(tmp_path / name), cfg, w))
        assert c.architecture == "Tikalix" and c.to_dict() == config_from_dict(c.to_dict()).to_dict()
        assert c.residual_mult == cfg.get("residual_mult", 1.0) and c.embedding_scale == cfg.get("embedding", {}).get("scale", 1.0)
        spec = ARCHITECTURES.get(c.architecture).build_spec(c)
        assert spec_tensors(spec) == {n: tuple(t.shape) for n, t in w.items()}
        assert len(spec.stages[0].calls) == len(spec.layers) == len(cfg["layers"])
        for layer, entry in zip(spec.layers, cfg["layers"]):
            assert ("feed_forward" in layer.parts) == (entry["mlp"] is not None) == ("feed_forward_post_norm" in layer.parts)
            assert layer.params["mult"] == cfg.get("residual_mult", 1.0)


def test_a_norm_around_an_absent_feed_forward_may_stay_in_the_file(tmp_path):
    cfg = TM.CONFIGS["A"]
    w = TM.random_weights(cfg, 1)
    w["l2.norm2"] = torch.zeros(cfg["width"], dtype=torch.bfloat16)
    eng = Engine(TM.write_folder(str(tmp_path / "m"), cfg, w), dtype="float32", max_tokens=64, max_requests=1, ops=TorchOps())
    assert torch.isfinite(eng.step([("a", [1, 2, 3], [2])]).logits).all()


def test_configuration_errors_name_the_key():
    good = TM.CONFIGS["A"]
    for path, value, word in [(("layers", 0, "type"), "mamba2", "type"), (("layers", 0, "mixer", "kv_heads"), 3, "kv_heads"),
                              (("layers", 0, "mixer", "rot", "dims"), 3, "rot.dims"), (("layers", 0, "mixer", "rot", "dims"), 22, "rot.dims"),
                              (("layers", 0, "mixer", "rot", "scaling", "fast"), 0.0, "scaling"),
                              (("layers", 0, "mixer", "rot", "scaling", "original"), "long", "original"),
                              (("layers", 0, "mixer", "rot", "base"), 1.0, "base"), (("layers", 0, "mixer", "softcap"), -1.0, "softcap"),
                              (("layers", 0, "mixer", "vdim"), 0, "vdim"), (("layers", 1, "mlp", "router", "top"), 9, "top"),
                              (("layers", 1, "mlp", "expert", "limit"), 0.0, "limit"), (("layers", 1, "mlp", "shared", "ff"), 0, "shared"),
                              (("layers", 0, "mlp", "kind"), "gated", "mlp"), (("norm",), {}, "eps"), (("residual_mult",), "x", "residual_mult")]:
        bad = copy.deepcopy(good)
        d = bad
        for k in path[:-1]:
            d = d[k]
        d[path[-1]] = value
        with pytest.raises(ConfigError, match=word):
            config_from_dict(bad)


# ---- the plain implementation's mechanisms against closed forms ----------------------------------------------------

def test_plain_rotation_and_its_slowed_waves():
    sc = {"factor": 4.0, "original": 64, "fast": 2.0, "slow": 0.5}
    f0, one = pt.rotary_frequencies(16, 1000.0)
    f, factor = pt.rotary_frequencies(16, 1000.0, sc)
    assert one == 1.0 and abs(factor - (0.1 * math.log(4.0) + 1.0)) < 1e-15
    # where a pair that turns `fast` (`slow`) times within `original` positions would sit: there the wave is original / turns long
    at = [16 * math.log(64 / (2 * math.pi * t)) / (2 * math.log(1000.0)) for t in (2.0, 0.5)]
    for a, t in zip(at, (2.0, 0.5)):
        assert abs(2 * math.pi / 1000.0 ** (-2 * a / 16) - 64 / t) < 1e-9
    lo, hi = math.floor(at[0]), math.ceil(at[1])
    assert 0 < lo < hi - 1 and hi < 7                           # all three kinds of pairs are there
    for i in range(8):
        if i <= lo:
            assert f[i] == f0[i]
        elif i >= hi:
            assert torch.isclose(f[i], f0[i] / 4.0, rtol=1e-14)
        else:
            r = (i - lo) / (hi - lo)
            assert torch.isclose(f[i], f0[i] * ((1 - r) + r / 4.0), rtol=1e-14) and f0[i] / 4 < f[i] < f0[i]
    # the engine's table is the same function written another way, also where both ends fall together or off the table
    for dims, base, args in ((16, 1000.0, (4.0, 64, 2.0, 0.5)), (64, 1e5, (4.0, 256, 8.0, 1.0)), (2, 1e4, (1.0, 16, 1.0, 1.0)),
                             (10, 300.0, (8.0, 32, 4.0, 1.0)), (8, 50.0, (3.0, 8, 1e-4, 1e-6)), (8, 50.0, (3.0, 8, 1e6, 1e4))):
        ours, c = pt.rotary_frequencies(dims, base, dict(zip(("factor", "original", "fast", "slow"), args)))
        theirs, d = slowed_frequencies(dims, base, *args)
        assert torch.allclose(ours, theirs, rtol=1e-13) and abs(c - d) < 1e-15
    # a pair's scalar product depends on the distance alone; channel i turns with channel i + dims/2; the rest stays
    torch.manual_seed(0)
    x, y = torch.randn(1, 1, 10, dtype=F64).expand(3, 1, 10), torch.randn(1, 1, 10, dtype=F64).expand(3, 1, 10)
    fr, _ = pt.rotary_frequencies(6, 50.0)
    a, b = pt.rotate_half(x, torch.tensor([3, 10, 40]), 6, fr), pt.rotate_half(y, torch.tensor([1, 8, 38]), 6, fr)
    s = (a * b).sum(-1)
    assert torch.allclose(s, s[0].expand(3, 1), atol=1e-12) and torch.equal(a[..., 6:], x[..., 6:])
    ang = 40 * 50.0 ** (-2.0 / 6)
    assert torch.isclose(a[2, 0, 1], x[2, 0, 1] * math.cos(ang) - x[2, 0, 4] * math.sin(ang), atol=1e-12)
    assert torch.isclose(a[2, 0, 4], x[2, 0, 4] * math.cos(ang) + x[2, 0, 1] * math.sin(ang), atol=1e-12)
    c = pt.rotate_half(x, torch.tensor([3, 10, 40]), 6, fr, factor=1.25)
    assert torch.allclose(c[..., :6], 1.25 * a[..., :6], atol=1e-12) and torch.equal(c[..., 6:], x[..., 6:])


def test_plain_attention_key_by_key():
    torch.manual_seed(1)
    T, W, eps = 7, 10, 1e-3
    m = {"heads": 4, "kv_heads": 2, "dim": 6, "vdim": 3, "scale": 0.9, "softcap": 2.0,
         "rot": {"dims": 4, "base": 20.0, "scaling": {"factor": 3.0, "original": 16, "fast": 2.0, "slow": 0.5}}}
    t = {"q": torch.randn(24, W), "q.b": torch.randn(24), "k": torch.randn(12, W), "k.b": torch.randn(12), "v": torch.randn(6, W),
         "v.b": torch.randn(6), "g": torch.randn(12, W), "o": torch.randn(W, 12)}
    t = {k: v.double() for k, v in t.items()}
    h = torch.randn(T, W, dtype=F64)
    got = pt.attention(h, t, "", m, eps, torch.arange(T))
    fr, factor = pt.rotary_frequencies(4, 20.0, m["rot"]["scaling"])

    def head(row, pos, name, i):
        u = (t[name][6 * i:6 * i + 6] @ h[row]) + t[name + ".b"][6 * i:6 * i + 6]
        r = u.clone()
        for j in range(2):
            c, s = math.cos(pos * fr[j]) * factor, math.sin(pos * fr[j]) * factor
            r[j], r[j + 2] = u[j] * c - u[j + 2] * s, u[j + 2] * c + u[j] * s
        return r / math.sqrt(float((r * r).sum()) / 6 + eps)                 # the norm comes after the rotation

    out = torch.zeros(T, 4, 3, dtype=F64)
    for i in range(T):
        for hd in range(4):
            e = [math.exp(2.0 * math.tanh(float(head(i, i, "q", hd) @ head(j, j, "k", hd // 2)) * 0.9 / 2.0)) for j in range(i + 1)]
            for j in range(i + 1):
                g = hd // 2
                out[i, hd] += e[j] / sum(e) * (t["v"][3 * g:3 * g + 3] @ h[j] + t["v.b"][3 * g:3 * g + 3])
    gate = 1.0 / (1.0 + torch.exp(-(h @ t["g"].T)))
    assert torch.allclose(got, (out.reshape(T, 12) * gate) @ t["o"].T, atol=1e-12)
    # weights add up to one, and no score leaves the cap
    w = pt.softmax_weights(torch.randn(5, 2, 4, dtype=F64) * 9, torch.randn(5, 1, 4, dtype=F64) * 9, 1.0, 2.0, pt.causal_mask(5))
    assert torch.allclose(w.sum(-1), torch.ones(2, 5, dtype=F64)) and (w.triu(1) == 0).all()
    assert all(float(row.max() / row.min()) <= math.exp(4.0) + 1e-9 for row in w[:, 4])
    assert torch.equal(pt.capped(torch.tensor([3.0, -70.0]), 0.0), torch.tensor([3.0, -70.0]))


def test_plain_choice_experts_and_clamps():
    z = torch.tensor([[0.5, 2.0, -1.0, 1.5], [-3.0, -2.0, -4.0, -200.0]], dtype=F64)
    ids, w, margins = pt.choose(z, 2)
    assert ids.tolist() == [[1, 3], [1, 0]]
    a = math.exp(2.0) / (math.exp(2.0) + math.exp(1.5))
    assert torch.allclose(w[0], torch.tensor([a, 1 - a], dtype=F64)) and torch.allclose(w.sum(-1), torch.ones(2, dtype=F64))
    assert margins == [1.0, 1.0] and pt.choose(z, 4)[2] == []
    torch.manual_seed(4)
    W = 6
    mlp = {"expert": {"ff": 5, "limit": 0.7}, "router": {"experts": 4, "top": 2}, "shared": {"ff": 3, "limit": 0.4}}
    t = {"router": torch.randn(4, W) * 2, "shared.gate": torch.randn(3, W), "shared.up": torch.randn(3, W), "shared.down": torch.randn(W, 3)}
    for e in range(4):
        t[f"e{e}.gate"], t[f"e{e}.up"], t[f"e{e}.down"] = torch.randn(5, W), torch.randn(5, W), torch.randn(W, 5)
    t = {k: v.double() for k, v in t.items()}
    h = torch.randn(9, W, dtype=F64)

    def expert(x, pre, limit):
        g = torch.minimum(x @ t[pre + "gate"].T, torch.tensor(limit, dtype=F64))
        u = torch.maximum(torch.minimum(x @ t[pre + "up"].T, torch.tensor(limit, dtype=F64)), torch.tensor(-limit, dtype=F64))
        return (g / (1 + torch.exp(-1.702 * g)) * (u + 1)) @ t[pre + "down"].T

    want = torch.zeros_like(h)
    for r in range(9):
        top = torch.topk(h[r] @ t["router"].T, 2)
        e = torch.exp(top.values)
        for k, i in enumerate(top.indices.tolist()):
            want[r] += e[k] / e.sum() * expert(h[r], f"e{i}.", 0.7)
    want = want + expert(h, "shared.", 0.4)
    assert torch.allclose(pt.moe_ff(h, t, "", mlp), want, atol=1e-12)
    z = h @ t["e0.gate"].T, h @ t["e0.up"].T
    assert (z[0] > 0.7).any() and (z[1] < -0.7).any() and (z[1] > 0.7).any()                # the clamps bit
    x = torch.tensor([[-1.0, 0.5, 2.0]], dtype=F64)
    assert torch.allclose(pt.dense_ff(x, {"up": torch.eye(3, dtype=F64), "down": torch.eye(3, dtype=F64)}, ""),
                          torch.tensor([[0.0, 0.25, 4.0]], dtype=F64))


def test_plain_norm_is_stored_around_zero():
    x = torch.tensor([[3.0, -4.0]], dtype=F64)
    r = math.sqrt(12.5 + 0.1)
    assert torch.allclose(pt.rms_norm(x, torch.tensor([0.0, 0.5], dtype=F64), 0.1), torch.tensor([[3.0 / r, -4.0 / r * 1.5]], dtype=F64))


# ---- the engine on the stand-ins against the plain implementation ---------------------------------------------------

@pytest.mark.parametrize("name", list(TM.CONFIGS))
def test_schedules_on_the_stand_in(name):
    cfg, w, w64 = model(name)
    reqs = {f"r{i}": H.random_ids(cfg["vocab"], n, 40 + i) for i, n in enumerate([37, 1, 58, 23, 70])}
    eng = engine_for(cfg, w)
    for steps in (H.whole_trace(reqs), H.tail_decode_trace(reqs, tail=12), H.portions_trace(reqs, seed=3)):
        got = TM.run_trace(eng, steps)
        assert len(got) == sum(len(v) for v in reqs.values())
        worst = TM.worst_error(name, cfg, w64, reqs, got)
        assert worst[0] <= TOL_OF.get(name, TOL32), worst
        assert eng.cache.n_live == 0
        eng.cache.check()
    # several requests at a time with pages for the live ones only: pages and slots are used again
    steps, peak = H.mixed_trace(reqs, max_live=3, seed=4)
    eng = engine_for(cfg, w, max_requests=3, max_tokens=peak, graphs=True)
    got = TM.run_trace(eng, steps)
    worst = TM.worst_error(name, cfg, w64, reqs, got)
    assert worst[0] <= TOL_OF.get(name, TOL32), worst
    eng.cache.check()


def test_the_stream_after_every_layer():
    """What the blocks leave in the 32-bit stream, layer by layer (also behind a layer without a feed-forward)."""
    for name in ("A", "B", "E"):
        cfg, w, w64 = model(name, seed=4)
        ids = H.random_ids(cfg["vocab"], 19, 3)
        want = []
        pt.forward(cfg, w64, ids, layers_out=want)
        eng = engine_for(cfg, w)
        seen = []
        for layer in eng.model.layers:
            def spy(x, ctx, run=layer.forward):
                y = run(x, ctx)
                seen.append(y.full.clone())
                return y
            layer.forward = spy
        eng.step([("s", ids, [len(ids) - 1])])
        assert len(seen) == len(want)
        for a, b in zip(seen, want):
            assert (a[:len(ids)].double() - b).abs().max() <= 3e-5 * b.abs().max()


def needle_case(name, at, distance, seed=60):
    """A sequence in which the probe token, `distance` after the needle at `at`, looks for it in the first layer; and how far
    the probe's logits move when the needle is replaced."""
    cfg, w, _ = model(name)
    cfg, w = TM.sharpen(cfg, w, 3, 7, distance)
    w64 = TM.as_f64(w)
    ids = [t if t not in (3, 7) else 11 for t in H.random_ids(cfg["vocab"], at + distance + 4, seed + at)]
    ids[at], ids[at + distance] = 3, 7
    without = list(ids)
    without[at] = 11
    key = (name, "sharp", distance)
    moved = TM.relative_error(pt.forward(cfg, w64, without)[at + distance], TM.plain_logits(key, cfg, w64, ids)[at + distance])
    return key, cfg, w, w64, ids, moved


@pytest.mark.parametrize("name,distance", [("A", 1), ("C", 300), ("B", 60), ("E", 130)])
def test_a_token_that_stands_out(name, distance):
    """The probe looks for a needle right before it or hundreds of tokens back, with the needle at the first position and on
    both sides of a page's border; whole, decoded alone and in portions."""
    for at in (0, 15, 16):
        key, cfg, w, w64, ids, moved = needle_case(name, at, distance)
        assert moved >= 0.05, moved              # losing that one key would show
        eng = engine_for(cfg, w)
        for steps in (H.whole_trace({"s": ids}), H.tail_decode_trace({"s": ids}, tail=6), H.portions_trace({"s": ids}, sizes=(5, 2, 11))):
            worst = TM.worst_error(key, cfg, w64, {"s": ids}, TM.run_trace(eng, steps))
            assert worst[0] <= TOL32, worst


def test_the_first_tokens_and_one_token_alone():
    for name in ("A", "B", "D"):
        cfg, w, w64 = model(name, seed=7)
        eng = engine_for(cfg, w)
        reqs = {"one": H.random_ids(cfg["vocab"], 1, 1), "two": H.random_ids(cfg["vocab"], 2, 2), "five": H.random_ids(cfg["vocab"], 5, 3)}
        for steps in (H.whole_trace(reqs), H.tail_decode_trace(reqs, tail=4)):
            got = TM.run_trace(eng, steps)
            assert TM.worst_error((name, 7), cfg, w64, reqs, got)[0] <= TOL_OF.get(name, TOL32)


def test_long_decoding_of_unequal_requests():
    """Three requests of unequal lengths decode 90 tokens together, over many page borders, each against itself alone."""
    cfg, w, w64 = model("A", seed=6)
    reqs = {f"r{i}": H.random_ids(cfg["vocab"], n, 90 + i) for i, n in enumerate([100, 131, 93])}
    eng = engine_for(cfg, w, max_requests=3, graphs=True)
    steps = [{"step": 0, "entries": [{"id": r, "tokens": ids[:len(ids) - 90], "want": [0]} for r, ids in reqs.items()], "end": []}]
    for t in range(90):
        steps.append({"step": t + 1, "entries": [{"id": r, "tokens": [ids[len(ids) - 90 + t]], "want": [0]} for r, ids in reqs.items()],
                      "end": list(reqs) if t == 89 else []})
    got = TM.run_trace(eng, steps)
    assert TM.worst_error(("A", 6), cfg, w64, reqs, got)[0] <= TOL32


def test_what_the_design_fixes_shows_in_the_logits(monkeypatch):
    """Each mechanism changed in the plain implementation moves its logits by more than 100 times the engine's tolerance: the
    schedules above would catch any of them."""
    cfg, w, w64 = model("A")
    ids = H.random_ids(cfg["vocab"], 40, 9)
    want = TM.plain_logits("A", cfg, w64, ids)

    def shows(what, changes, cfg=cfg):
        with monkeypatch.context() as mp:
            for name, fn in changes.items():
                mp.setattr(pt, name, fn)
            assert TM.relative_error(pt.forward(cfg, w64, ids)[20], want[20]) > 100 * TOL32, what

    unit, rotate, freqs, expert, choose = pt.unit_rms, pt.rotate_half, pt.rotary_frequencies, pt.clamped_expert, pt.choose
    shows("no cap", {"capped": lambda s, cap: s})
    shows("weights stored as gains", {"rms_norm": lambda x, w_, eps: unit(x, eps) * w_})
    shows("queries and keys as they are", {"unit_rms": lambda x, eps: x if x.dim() == 3 else unit(x, eps)})

    def before(x, positions, dims, f, factor=1.0):        # unit length before the rotation instead of after it
        return rotate(unit(x, 1e-5), positions, dims, f, factor)
    shows("unit before rotation", {"rotate_half": before, "unit_rms": lambda x, eps: x if x.dim() == 3 else unit(x, eps)})
    shows("no factor on cosine and sine", {"rotary_frequencies": lambda *a: (freqs(*a)[0], 1.0)})
    shows("no slowed waves", {"rotary_frequencies": lambda d, b, s=None: (freqs(d, b)[0], freqs(d, b, s)[1])})

    def over_all(z, top):
        ids_, _, mg = choose(z, top)
        return ids_, torch.gather(torch.softmax(z, -1), 1, ids_), mg
    shows("a softmax over all experts", {"choose": over_all})
    shows("no clamp", {"clamped_expert": lambda h, w_, pre, limit: expert(h, w_, pre, 1e9)})
    shows("no shared expert", {"clamped_expert": lambda h, w_, pre, limit: expert(h, w_, pre, limit) * (0.0 if "shared" in pre else 1.0)})
    other = copy.deepcopy(cfg)
    other["residual_mult"] = 1.0
    shows("no factor on the branches", {}, other)
    other = copy.deepcopy(cfg)
    del other["embedding"]
    shows("no scale on the embedding", {}, other)
    flat = {n: (torch.zeros_like(t) if n.endswith("mix.g") else t) for n, t in w64.items()}
    assert TM.relative_error(pt.forward(cfg, flat, ids)[20], want[20]) > 100 * TOL32


def test_greedy_generation_through_the_scheduler():
    for name in ("A", "B"):
        cfg, w, w64 = model(name, seed=8)
        prompts = [H.random_ids(cfg["vocab"], n, 80 + i) for i, n in enumerate((13, 1, 30, 6))]
        want = [pt.greedy_generate(cfg, w64, p, 7) for p in prompts]
        eng = engine_for(cfg, w, max_requests=2, max_tokens=160, graphs=True)
        out, s = generate(eng, prompts, max_new_tokens=7, temperature=0.0, max_batch=2, token_budget=11,
                          return_scheduler=True)
        assert out == want
        assert s.peak_running == 2 and eng.cache.n_live == 0
        eng.cache.check()


def test_the_named_size_runs_with_random_weights(tmp_path):
    from tiny_inference_server_amd.__main__ import preset_names, size_config
    from tiny_inference_server_amd.weights import write_random_model
    assert "tikalix-small" in preset_names()
    cfg = size_config("tikalix-small")
    folder = write_random_model(cfg, 3, str(tmp_path / "m"))
    assert load_config(folder).to_dict() == cfg.to_dict()
    eng = Engine(folder, dtype="float32", max_tokens=64, max_requests=2, ops=TorchOps())
    out = eng.step([("a", [5, 9, 1, 300], [3]), ("b", [7], [0])]).logits
    assert out.shape == (2, cfg.vocab) and torch.isfinite(out).all()


class PlannedOps(TorchOps):
    """The stand-in with the device's own attention planning, whose lists it carries through every step and ignores."""

    def plan_attention_mode(self, seq_rows, window=0):
        return HipOps.plan_attention_mode(SimpleNamespace(dtype=torch.bfloat16), seq_rows, window)

    def plan_attention(self, *args, **kw):
        return HipOps.plan_attention(SimpleNamespace(dtype=torch.bfloat16, units=256), *args, **kw)


@pytest.mark.parametrize("sizes", [((4, 2, 20, 20, 30.0), (4, 2, 20, 20, None)), ((4, 2, 20, 24, None), (4, 2, 20, 24, 6.0), (4, 2, 20, 24, 2.0)),
                                   ((4, 2, 20, 20, 6.0), (4, 2, 32, 32, 6.0)), ((6, 3, 16, 48, None), (6, 3, 32, 32, None), (6, 3, 48, 16, None))])
@pytest.mark.parametrize("lengths", [(9,), (300, 20, 25, 30, 18, 22, 27, 19, 31, 26, 24, 23)])
def test_layers_that_differ_in_caps_or_head_sizes_alone_decode_from_captured_steps(sizes, lengths):
    """A captured step must find a place for every list that is planned for the step after, whether layers share one or not. One request, and requests of
    such different lengths that their splits are planned."""
    cfg = TM.config(48, 97, [TM.layer(TM.mixer(H_, G, D, V, 0.4, cap=cap, dims=8), TM.dense(24)) for H_, G, D, V, cap in sizes])
    c, w = config_from_dict(cfg), {n: t.float() for n, t in TM.random_weights(cfg, 3).items()}
    replayed, launched = (Engine(config=c, tensors=w, dtype="float32", page_size=16, max_tokens=2048, max_requests=len(lengths), use_graphs=graphs, ops=PlannedOps(graphs=graphs))
                          for graphs in (True, False))
    ids = {f"r{i}": H.random_ids(97, n + 8, 40 + i) for i, n in enumerate(lengths)}
    for eng in (replayed, launched):
        for rid, t in ids.items():
            eng.step([(rid, t[:-8], [])])
    for k in range(8):
        entries = [(rid, [t[len(t) - 8 + k]], [0]) for rid, t in ids.items()]
        got, want = replayed.step(entries).logits, launched.step(entries).logits
        assert (got - want).abs().max().item() <= 1e-5 * max(1.0, want.abs().max().item())
    assert replayed.graph_replays >= 6
    if len(lengths) > 1:
        assert any(g.mode is not None for g in replayed._graphs.values())
