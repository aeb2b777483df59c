"""The names that attention's planned lists go by: whoever plans for the launch uses the ones that the launch looks for."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from test_product_routes import host_ops
from tiny_inference_server_amd.ops import kernel_bench


@pytest.mark.parametrize("segments,mode", [("100:1x3,0:40", None), ("0:300", None), ("4000:1x8,10:1x24", "uneven"), ("4000:1,10:1x3,0:700", None)])
@pytest.mark.parametrize("heads,kv_heads,dim", [(4, 2, 64), (12, 3, 128)])
def test_the_measurement_tool_plans_as_the_engine_does(monkeypatch, capsys, segments, mode, heads, kv_heads, dim):
    seen = []
    monkeypatch.setattr(kernel_bench, "graph_time", lambda fn, reps: fn() or 1.0)
    tool = SimpleNamespace(device="cpu", units=256, paged_attention=lambda q, plane, batch, *args: seen.append(batch))
    kernel_bench.attention_case(tool, SimpleNamespace(heads=heads, kv_heads=kv_heads, head_dim=dim, page_size=16, segments=segments, planned=False,
                                                      same_splits=False, no_tiles=False, tiles=False, reps=1))
    packed = []
    engine = host_ops()
    engine.units = tool.units
    plans = engine.plan_attention(heads, kv_heads, dim, seen[0].seq_rows, lambda array: packed.append(array) or len(packed) - 1, mode)
    lists = {name: made for name, made in plans.items() if name[0] != "attention_tile_pieces"}
    assert set(seen[0].extras) == set(lists) and len(lists) == 1
    name, made = lists.popitem()
    assert seen[0].extras[name][1:] == made[1:]
    assert torch.equal(seen[0].extras[name][0], torch.from_numpy(packed[made[0]]).reshape(-1))
