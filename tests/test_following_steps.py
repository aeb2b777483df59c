"""The step that a replayed step of single tokens prepares: taken when the same requests come again in the same order, and only then."""
from __future__ import annotations

import pytest
import torch

import helpers as H
from tiny_inference_server_amd.cache.manager import OutOfPages
from tiny_inference_server_amd.engine import Engine
from torch_ops import TorchOps


def engine(n, max_tokens=640):
    folder = H.model_folder("A", "float32")
    eng = Engine(folder, dtype="float32", page_size=16, max_tokens=max_tokens, max_requests=n, ops=TorchOps(graphs=True))
    taken = []
    inner = eng._run_following
    eng._run_following = lambda f, tokens: (taken.append(len(tokens)), inner(f, tokens))[1]
    return folder, eng, taken


@pytest.mark.parametrize("n", [1, 3, 11])
def test_prepared_steps_give_what_each_request_alone_gives(n):
    """Requests that open pages at different steps (16 positions a page), up to filled-up shapes; now and then in another order, without one of
    them, with a step of another kind between: every logit is the plain model's."""
    vocab = H.TINY["A"]["cfg"].vocab_size
    folder, eng, taken = engine(n, max_tokens=80 * n)
    ids = {f"r{i}": H.random_ids(vocab, 60, 700 + i) for i in range(n)}
    at = {r: 9 + i % 7 for i, r in enumerate(ids)}
    for r, t in ids.items():
        eng.step([(r, t[:at[r]], [])])
    main = {}
    for k in range(30):
        order = list(ids)
        if k in (8, 9):
            order = order[::-1]
        if k == 15 and n > 1:
            order = order[:-1]
        portion = 2 if k == 20 else 1
        entries = [(r, ids[r][at[r]:at[r] + portion], [portion - 1]) for r in order]
        out = eng.step(entries, heads=k == 24)
        for r, lg in zip(order, out.logits):
            at[r] += portion
            main[(r, at[r] - 1)] = lg.clone()
    assert len(taken) >= 15 and set(taken) <= {n, max(1, n - 1)}
    worst = 0.0
    for r, t in ids.items():
        want = H.plain_logits(folder, t)[0]
        for (q, p), got in main.items():
            if q == r:
                worst = max(worst, (got.double() - want[p]).abs().max().item() / max(1.0, want.abs().max().item()))
    assert worst <= 2e-5
    eng.cache.check()


def test_what_is_wrong_with_a_step_is_said_as_ever():
    vocab = H.TINY["A"]["cfg"].vocab_size
    folder, eng, taken = engine(2, max_tokens=64)
    for r in ("a", "b"):
        eng.step([(r, H.random_ids(vocab, 10, 5), [])])
    one = lambda t=1: [("a", [t], [0]), ("b", [2], [0])]
    for _ in range(4):
        eng.step(one())
    assert eng._following is not None and taken
    with pytest.raises(ValueError, match="outside the vocabulary"):
        eng.step(one(vocab))
    with pytest.raises(ValueError):
        eng.step([("a", [1], [1]), ("b", [2], [0])])
    with pytest.raises(ValueError, match="twice"):
        eng.step([("a", [1], [0]), ("a", [2], [0])])
    assert eng.fed("a") == eng.fed("b") == 14
    eng.step([("a", [1], iter([0])), ("b", [2], {0})])      # places wanted as anything that can be walked
    assert eng.fed("a") == eng.fed("b") == 15
    eng.reserve("a", 40)                     # takes a page the step was not prepared for
    eng.step(one())
    with pytest.raises(OutOfPages):          # four pages in all: b cannot open its second and a third
        for _ in range(60):
            eng.step(one())
    fed = eng.fed("b")
    eng.close("a")
    eng.step([("b", [3], [0])])
    assert eng.fed("b") == fed + 1
    eng.cache.check()


def test_a_prepared_step_is_not_replayed_once_replays_are_switched_off():
    """use_decode_graphs is read at every step, also at one that was prepared while it was still on."""
    vocab = H.TINY["A"]["cfg"].vocab_size
    folder, eng, taken = engine(1)
    ids = H.random_ids(vocab, 20, 9)
    eng.step([("a", ids[:10], [])])
    for p in range(10, 14):
        eng.step([("a", ids[p:p + 1], [0])])
    assert eng._following is not None and taken
    steps, replays = len(taken), eng.graph_replays
    eng.use_decode_graphs = False
    out = eng.step([("a", ids[14:15], [0])])
    assert len(taken) == steps and eng.graph_replays == replays
    want = H.plain_logits(folder, ids)[0][14]
    assert (out.logits[0].double() - want).abs().max().item() <= 2e-5 * max(1.0, want.abs().max().item())
    eng.use_decode_graphs = True
    for p in range(15, 18):
        eng.step([("a", ids[p:p + 1], [0])])
    assert eng.graph_replays > replays and len(taken) > steps
