"""Prepared steps of a model with windows beside full attention, and of a batch whose work lists come and go: the branches of the step after a replayed
one that a small batch of one page group never sees."""
from __future__ import annotations

import dataclasses

import pytest
import torch

import helpers as H
from tiny_inference_server_amd.architectures.gqa_mtp import _block, _norm
from tiny_inference_server_amd.config import ARCHITECTURES, Architecture, GqaMtpConfig
from tiny_inference_server_amd.engine import Engine
from tiny_inference_server_amd.parts import LayerCall, ModelSpec, PartSpec, StageSpec
from tiny_inference_server_amd.ops import hip_ops
from tiny_inference_server_amd.weights import random_tensors
from torch_ops import TorchOps

WINDOWS = (24, 0, 40)


class PlanningOps(TorchOps):
    """The stand-in with the attention mixer's planning of uneven single rows, by window, as the device's operations have it; its attention ignores
    the lists."""

    def plan_attention_mode(self, seq_rows, window=0):
        return "uneven" if hip_ops.uneven_lengths(seq_rows, window) else None

    def plan_attention(self, n_heads, n_kv_heads, head_dim, seq_rows, add, mode=None, window=0):
        if mode != "uneven":
            return {}
        entries, most = hip_ops.decode_items(seq_rows, n_heads, n_kv_heads, head_dim, window=window)
        return {("attention_decode_items", n_heads, n_kv_heads, window): (add(entries), len(entries), most)}


@pytest.fixture(scope="module")
def model():
    """Three layers, two of which see the last keys only: three page groups."""
    def spec(cfg):
        layers = []
        for l, window in enumerate(WINDOWS):
            block = _block(cfg, f"transformer_block_list.{l}.")
            mixer = block.part("mixer")
            layers.append(block.with_part("mixer", dataclasses.replace(mixer, params={**mixer.params, "window": window})))
        stage = StageSpec("trunk", 0, PartSpec("stage_input", "token_embedding"), tuple(LayerCall(l) for l in range(len(WINDOWS))),
                          _norm(cfg, "rms_out.scale"))
        return ModelSpec(cfg.d_model, cfg.vocab_size, cfg.max_context, tuple(layers), (stage,), "embedding.weight", "embedding.weight")
    name = "PreparedStepsToy"
    ARCHITECTURES.register(name, Architecture(name, GqaMtpConfig, spec), replace=True)
    cfg = GqaMtpConfig(d_model=128, vocab_size=211, max_context=512, rope_base=1e4, n_heads=4, n_layers=3, ffn_hidden=160, group_size=2, mtp_heads=0,
                       architecture=name)
    yield cfg
    ARCHITECTURES.unregister(name)


@pytest.mark.parametrize("backend", [pytest.param("hip", marks=pytest.mark.gpu), "torch"])
@pytest.mark.parametrize("dtype,tol", [("float32", 2e-5), ("bfloat16", 4e-2)])
@pytest.mark.parametrize("table_pages", [64, 3])
def test_windows_plans_and_tables_of_prepared_steps(model, dtype, tol, backend, table_pages):
    """Eighteen requests, one of them long at first, decode side by side: their splits are planned request by request until the others have
    caught up, they open pages at different steps, give pages back behind their windows, and (table_pages 3) outgrow the captured tables. Every
    logit against an engine that launches every step, most of them from steps that were prepared, planned and not."""
    if backend == "torch" and dtype == "bfloat16":
        pytest.skip("the stand-in runs this in 32 bits")
    weights = random_tensors(model, 21, std=0.08, gain_jitter=0.1, dtype=dtype)
    make = lambda graphs: Engine(config=model, tensors=weights, dtype=dtype, page_size=16, max_tokens=16 * 110, max_requests=18, use_graphs=graphs,
                                 ops=PlanningOps(graphs=graphs) if backend == "torch" else None)
    replayed, launched = make(True), make(False)
    assert len(replayed.cache.groups) == 3 and not launched.use_decode_graphs
    replayed.graph_table_pages = table_pages
    taken, inner = [], replayed._run_following
    replayed._run_following = lambda f, tokens: (taken.append((f.graph.mode is not None, f.graph.table_at[next(iter(f.graph.table_at))][1][1], bool(f.opening))),
                                                 inner(f, tokens))[1]
    steps = 56
    ids = {f"r{i}": H.random_ids(model.vocab_size, (100 if i == 4 else 9 + i) + steps, 300 + i) for i in range(18)}
    for eng in (replayed, launched):
        for r, t in ids.items():
            eng.step([(r, t[:-steps], [])])
    for k in range(steps):
        entries = [(r, [t[len(t) - steps + k]], [0]) for r, t in ids.items()]
        got, want = replayed.step(entries).logits.float(), launched.step(entries).logits.float()
        assert (got - want).abs().max().item() <= tol * max(1.0, want.abs().max().item()), k
        for eng in (replayed, launched):
            for r in ids:
                held = {name: group.held(eng.requests[r][0]) for name, group in eng.cache.groups.items()}
                assert held["kv2x32w24"] <= 24 // 16 + 2 and held["kv2x32w40"] <= 40 // 16 + 2
    assert launched.graph_replays == 0 and len(taken) >= 30
    # prepared steps with a plan (32 bits on the device plan nothing) and without, that open pages and not, and with tables of several widths
    plans = {planned for planned, _, _ in taken}
    assert plans == ({False} if backend == "hip" and dtype == "float32" else {False, True})
    assert {opening for _, _, opening in taken} == {False, True}
    assert len({width for _, width, _ in taken}) == (1 if table_pages == 64 else 2)
    for eng in (replayed, launched):
        eng.cache.check()
        for r in ids:
            eng.close(r)
        eng.cache.check()
        assert eng.cache.free_pages() == eng.cache.total_pages()
