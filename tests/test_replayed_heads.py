"""Prompts whose prediction heads' logits are asked for, replayed from their third occurrence on."""
from __future__ import annotations

import pytest
import torch

import helpers as H
from tiny_inference_server_amd.engine import Engine
from torch_ops import TorchOps


@pytest.mark.parametrize("name,dtype", [pytest.param("E", "bfloat16", marks=pytest.mark.gpu), pytest.param("A", "float32", marks=pytest.mark.gpu),
                                        pytest.param("A", "float32-torch")])
def test_replayed_heads_are_what_a_launched_step_gives(name, dtype):
    """Prompts of the same lengths again and again, other tokens each time, one of them too short for the last head's row; other steps and
    closed requests between. Every replay against an engine that launches every step: the same logits, the same rows that are not there yet,
    and what an earlier step returned stays as it was."""
    dtype, _, backend = dtype.partition("-")
    folder = H.model_folder(name, dtype)
    vocab = H.TINY[name]["cfg"].vocab_size
    make = lambda graphs: Engine(folder, dtype=dtype, page_size=16, max_tokens=1024, max_requests=4, use_graphs=graphs,
                                 ops=TorchOps(graphs=graphs) if backend else None)
    kept, plain = make(True), make(False)
    if not kept.model.max_lag:
        pytest.skip("a model without prediction heads")
    lengths, held = (70, 33, 1, 140), []
    for k in range(6):
        prompts = [H.random_ids(vocab, n, 31 * k + n) for n in lengths]
        entries = [(f"r{i}", t, [len(t) - 1]) for i, t in enumerate(prompts)]
        before = kept.graph_replays
        a, b = kept.step(entries, heads=True), plain.step(entries, heads=True)
        assert (kept.graph_replays > before) == (k >= 2)
        assert a.head_valid == b.head_valid and [False] in [[v[2]] for v in a.head_valid]
        held.append([(x, y.clone()) for x, y in zip([a.logits] + a.head_logits, [b.logits] + b.head_logits)])
        for e in (kept, plain):
            e.step([("r0", [5], [0]), ("r1", [6], [0])])
            for i in range(4):
                e.close(f"r{i}")
    for step in held:
        for x, y in step:
            assert torch.equal(torch.isnan(x), torch.isnan(y))
            torch.testing.assert_close(torch.nan_to_num(x), torch.nan_to_num(y), rtol=0, atol=2e-2 if dtype == "bfloat16" else 2e-5)


@pytest.mark.parametrize("name,dtype", [pytest.param("A", "float32", marks=pytest.mark.gpu), pytest.param("A", "float32-torch")])
def test_no_graph_goes_on_holding_logits_of_many_places(name, dtype):
    """Steps with the heads' logits whose logits pass max_heads_graph_bytes are launched however often their shape comes; one place fewer
    is captured. Same logits either way."""
    dtype, _, backend = dtype.partition("-")
    folder = H.model_folder(name, dtype)
    vocab = H.TINY[name]["cfg"].vocab_size
    eng = Engine(folder, dtype=dtype, page_size=16, max_tokens=256, max_requests=1, ops=TorchOps(graphs=True) if backend else None)
    ids = H.random_ids(vocab, 40, 3)
    eng.max_heads_graph_bytes = 4 * (1 + eng.model.max_lag) * 39 * vocab
    kept = []
    for places in (40, 39):
        for k in range(4):
            before = eng.graph_replays
            out = eng.step([("a", ids, list(range(40 - places, 40)))], heads=True)
            eng.close("a")
            kept.append([out.logits[-39:]] + [h[-39:] for h in out.head_logits])
            assert (eng.graph_replays > before) == (places == 39 and k >= 2)
    for step in kept[1:]:
        for x, y in zip(step, kept[0]):
            torch.testing.assert_close(torch.nan_to_num(x), torch.nan_to_num(y), rtol=0, atol=2e-5)
