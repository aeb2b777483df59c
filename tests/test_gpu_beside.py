"""A block's two mixers side by side on two streams against one after the other."""
from __future__ import annotations

import pytest
import torch

import fesupel_models
import fikevik_models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("family,name", [("fesupel", "C"), ("fikevik", "E"), ("fikevik", "A")])
@pytest.mark.parametrize("launched", [True, False])
def test_the_same_bits(family, name, launched, monkeypatch):
    """Portions around the rule's first row count, a long one beside single rows, and portions that go on from used state lines, several passes of each in a
    row, so that memory given back by one pass is taken by the next and that the later ones are replayed from captured graphs: the same kernels on the same
    operands, so the same bits."""
    from tiny_inference_server_amd.config import config_from_dict
    from tiny_inference_server_amd.engine import Engine
    from tiny_inference_server_amd.ops.hip_ops import _BESIDE_FROM, HipOps
    monkeypatch.setattr("tiny_inference_server_amd.ops.hip_ops._BESIDE_WIDTH", 1)        # (as many rows as a wide model, however narrow this one is)
    if launched:
        monkeypatch.setattr("tiny_inference_server_amd.ops.hip_ops._BESIDE_LAUNCHED_FROM", _BESIDE_FROM)
    if family == "fesupel":
        cfg = fesupel_models.CONFIGS[name]
        w = fesupel_models.random_weights(cfg, 5)
    else:
        cfg = fikevik_models.CONFIGS[name]
        w = fikevik_models.random_weights(cfg, fikevik_models.RANK[name], 5)
    vocab = cfg["vocab"]
    steps = [[("a", _BESIDE_FROM - 1)], [("b", _BESIDE_FROM)], [("a", 1), ("b", _BESIDE_FROM + 1), ("c", 300)], [("a", 200), ("b", 1), ("c", 2)], [("c", 700)]]
    counts, results = [], []
    inner = HipOps.beside
    monkeypatch.setattr(HipOps, "beside", lambda self, *a: (counts.append(1), inner(self, *a))[1])
    for beside in (True, False):
        if not beside:
            monkeypatch.setattr(HipOps, "beside_pays", lambda self, batch, width: False)
        eng = Engine(config=config_from_dict(cfg), tensors=w, dtype="bfloat16", max_requests=4, page_size=16, max_tokens=2048)
        g = torch.Generator().manual_seed(3)
        seen, ran = [], [{} for _ in range(5)]
        for turn in range(5):
            for entries in steps:
                before = len(counts)
                seen.append(eng.step([(r, torch.randint(0, vocab, (n,), generator=g).tolist(), [0, n - 1]) for r, n in entries]).logits.clone())
                ran[turn][min(max(n for _, n in entries), _BESIDE_FROM)] = len(counts) > before
            for r in "abc":
                eng.close(r)
        assert eng.graph_replays >= 3 * len(steps) - 1      # (from a shape's third occurrence on)
        assert [r[_BESIDE_FROM] for r in ran] == [beside and launched] * 2 + [beside, False, False] and not any(r[_BESIDE_FROM - 1] for r in ran)
        results.append(seen)
    assert all(torch.isfinite(y).all() for y in results[0])
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_a_captured_pass_does_not_keep_every_blocks_result():
    """Eight blocks in a row in a capture, whose side results of 64 MB each are dropped block by block: their memory is taken again within the capture, so that
    the graph's pool holds two at most and not eight; and every replay, with eager work in between, gives what the blocks give by themselves."""
    from tiny_inference_server_amd.ops.hip_ops import HipOps
    ops = HipOps("cuda:0", torch.bfloat16)
    n, blocks = 16 << 20, 8
    x = torch.randn(n, device="cuda")

    def passes():
        total = torch.zeros(1024, device="cuda")
        for i in range(blocks):
            here, there = ops.beside(lambda: x[:1024] * (i + 1.0), lambda: x + float(i))
            total = total + here + there[i * 1024:(i + 1) * 1024]
            del here, there
        return total

    want = passes().clone()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_reserved()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = passes()
    assert torch.cuda.memory_reserved() - before < 3 * 4 * n
    for _ in range(4):
        graph.replay()
        passes()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_the_side_stream_is_the_threads_own():
    """None of the streams that the framework hands out in turn, nor another running thread's; a thread that has ended leaves its stream to the next."""
    import threading

    from tiny_inference_server_amd.ops.hip_ops import _beside_stream
    others = {torch.cuda.Stream().cuda_stream for _ in range(40)}
    mine, seen, gone = _beside_stream(0), [], []

    def ask():
        seen.append(_beside_stream(0))
        y = torch.zeros(4, device="cuda")
        torch.cuda.synchronize()
        with torch.cuda.stream(seen[-1]):
            gone.append(float((y + 1).sum()))

    for _ in range(2):
        t = threading.Thread(target=ask)
        t.start()
        t.join()
    assert _beside_stream(0).cuda_stream == mine.cuda_stream not in others
    assert seen[0].cuda_stream == seen[1].cuda_stream not in others | {mine.cuda_stream}
    assert seen[0].priority == 0 and gone == [4.0, 4.0]
