"""Products of a model's own layers at the row counts of prompts: every tile of the tiled product, the gate taken on its sums, and
the choice between it and the library's product."""
from __future__ import annotations

import pytest
import torch

from tiny_inference_server_amd.ops import hip_ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    return hip_ops.HipOps("cuda:0", torch.bfloat16)


def rnd(shape, seed, std=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * std).to(torch.bfloat16)


# (rows, columns, inner) that take each tile: sizes that end inside a tile and inside a step
SIZES = {0: (2044, 8188, 1544), 1: (1020, 6148, 1032), 2: (1000, 4100, 1096), 3: (2049, 5160, 264), 4: (700, 4100, 1032), 5: (500, 2308, 1032),
         6: (300, 2052, 520), 7: (300, 1028, 520)}


@pytest.mark.parametrize("tile", sorted(SIZES))
def test_every_tile(ops, tile):
    """Against exact sums of the same operands: the 32-bit result within what 32-bit sums of K terms differ by, the others one rounding
    to bfloat16 further; the gate against the kernel that reads the stored product, to the bit."""
    M, N, K = SIZES[tile]
    assert ops.gemm_tiles.cdll.tis_gemm_tiles_pick(M, N, K) == tile
    x, w, res = rnd((M, K), 1).cuda(), rnd((N, K), 2, K ** -0.5).cuda(), rnd((M, N), 3).cuda()
    want = (x.double() @ w.double().t())
    torch.testing.assert_close(ops._linear_tiles(x, w, None, torch.empty(M, N, device="cuda"), N, 1, 0).double(), want, rtol=1e-4, atol=1e-4)
    out = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
    ops._linear_tiles(x, w, res, out[:M], N, 0, 0)
    torch.testing.assert_close(out[:M].double(), want + res.double(), rtol=8e-3, atol=4e-3)
    assert bool((out[M] == 7.0).all())                  # nothing behind the last row
    gated = ops._linear_tiles(x, w, None, torch.empty(M, N // 2, dtype=torch.bfloat16, device="cuda"), N, 0, 4)
    assert torch.equal(gated, ops.swiglu(ops._linear_tiles(x, w, None, torch.empty(M, N, dtype=torch.bfloat16, device="cuda"), N, 0, 0)))


@pytest.mark.parametrize("M", [129, 300, 1024, 1025])
def test_products_by_rows(ops, M):
    """Widths of the library's list and another: up to the limit the tiles, beyond it what linear takes. The same sums in the same order
    either way, so the same bits; a residual whose rows the library does not take, too."""
    for i, (N, K) in enumerate(((2304, 1536), (1536, 4096), (1000, 640))):
        x, w, res = rnd((M, K), 10 + i).cuda(), rnd((N, K), 20 + i, K ** -0.5).cuda(), rnd((M, N + 8), 30 + i).cuda()[:, 4:N + 4]
        gain = (1 + 0.1 * torch.randn(K, generator=torch.Generator().manual_seed(5))).cuda()
        want = x.double() @ w.double().t()
        torch.testing.assert_close(ops.linear_by_rows(x, w, residual=res).double(), want + res.double(), rtol=2e-2, atol=2e-2)
        whole = res.contiguous()
        assert torch.equal(ops.linear_by_rows(x, w, residual=whole), ops.linear(x, w, residual=whole))
        assert torch.equal(ops.linear_by_rows(x, w, rms=(gain, 1e-5)), ops.linear(x, w, rms=(gain, 1e-5)))
        assert torch.equal(ops.linear_swiglu(x, w, rms=(gain, 1e-5)), ops.swiglu(ops.linear(x, w, rms=(gain, 1e-5))))
