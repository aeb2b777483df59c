"""Small kernels that wait for memory more than they work: the arg-max."""
from __future__ import annotations

import pytest
import torch

from tiny_inference_server_amd.ops import hip_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [1, 3, 64, 1023, 4099, 24576, 24580, 24583, 48000, 100001])
def test_argmax(V):
    """The first of the largest values, wherever they lie: one row each for the ends of a thread's pieces and for ties; a row of -inf."""
    ops = hip_ops.HipOps("cuda:0", torch.float32)
    x = torch.randn(10, V, generator=torch.Generator().manual_seed(V)).clamp(max=2.0)       # (many ties at 2)
    for r, at in enumerate((0, V - 1, V // 2, min(V - 1, 4095), min(V - 1, 24575), min(V - 1, 24576))):
        x[r, at] = 9.0
    x[8, V // 3:] = 3.0
    x[9] = -float("inf")
    for shift in (0, 1):                                   # rows that start on 16 bytes, and rows that do not
        rows = torch.zeros(10, -(-V // 4) * 4 + 4 + shift, device="cuda")[:, shift:V + shift]
        rows.copy_(x)
        assert ops.argmax(rows).cpu().tolist()[:9] == x.argmax(-1).tolist()[:9]
