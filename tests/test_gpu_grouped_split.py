"""The grouped product of a few rows a group with its sum over K split over a workgroup's waves."""
from __future__ import annotations

from ctypes import c_long

import pytest
import torch

from tiny_inference_server_amd.ops import hip_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(1, 384), (15, 392), (16, 512), (17, 520), (64, 640), (65, 1024), (130, 1032), (48, 1544), (200, 4096)])
@pytest.mark.parametrize("rows,groups,top", [(1, 2, 1), (5, 9, 2), (16, 3, 3)])
def test_against_64_bits(N, K, rows, groups, top):
    """Column counts around a block of 16, sums that end inside a batch, groups without an entry, with some and with all rows, with and without the gate of pairs of columns,
    to both result types. Bound: K products of bfloat16 numbers, exact in 32 bits, added in any order are off by at most K 2^-24 of the sum of their
    sizes (here in chains of at most K / 4 + 20, so a quarter of that is given); a bfloat16 result by another 2^-9 of itself."""
    ops = hip_ops.HipOps("cuda:0", torch.bfloat16)
    g = torch.Generator().manual_seed(N + rows)
    x = torch.randn(rows, K, generator=g).bfloat16()
    w = (torch.randn(groups, N, K, generator=g) * K ** -0.5).bfloat16()
    chosen = torch.stack([torch.randperm(groups, generator=g)[:top] for _ in range(rows)])
    lists, counts = torch.full((groups, rows), 1 << 20, dtype=torch.int32), torch.zeros(groups, dtype=torch.int32)
    for r in range(rows):
        for k in range(top):
            e = int(chosen[r, k])
            lists[e, counts[e]] = r * top + k
            counts[e] += 1
    flat = chosen.reshape(-1)
    rows64 = x.double().repeat_interleave(top, 0)
    want = torch.einsum("ek,enk->en", rows64, w.double()[flat])
    size = torch.einsum("ek,enk->en", rows64.abs(), w.double()[flat].abs())
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.full((rows * top, N), 7.0, dtype=dtype, device="cuda")
        ops._grouped(x.cuda(), K, 0, top, w.cuda(), out, N, 0, lists.cuda(), counts.cuda(), rows, rows)
        got = out.double().cpu()
        bound = size * (K / 4) * 2.0 ** -24 + (want.abs() * 2.0 ** -8 if dtype == torch.bfloat16 else 0)
        assert ((got - want).abs() <= bound).all(), ((got - want).abs() / bound).max()
    if N % 2 == 0:
        limit = 0.8
        out = torch.full((rows * top, N // 2), 7.0, dtype=torch.float32, device="cuda")
        ops._grouped(x.cuda(), K, 0, top, w.cuda(), out, N // 2, 0, lists.cuda(), counts.cuda(), rows, rows, act=2, limit=limit)
        a, u = want[:, 0::2].clamp(max=limit), want[:, 1::2].clamp(-limit, limit)
        gated = a * torch.sigmoid(1.702 * a) * (u + 1)
        # (the gate's slope in its first argument is below 1.2 (u + 1), in its second at most `limit`; expf and the division add some 2^-21 of the result)
        bound = (size[:, 0::2] * 1.2 * (1 + limit) + size[:, 1::2] * limit) * (K / 4) * 2.0 ** -24 + gated.abs() * 2.0 ** -20 + 2.0 ** -24
        got = out.double().cpu()
        assert ((got - gated).abs() <= bound).all()


@pytest.mark.parametrize("N,K", [(1, 384), (16, 392), (17, 520), (65, 1032), (48, 1544)])
@pytest.mark.parametrize("rows,heads", [(1, 2), (16, 3), (17, 4), (40, 2)])
def test_a_product_per_head_against_64_bits(N, K, rows, heads):
    """Groups of all rows, their columns apart in inputs and results, with and without a gate: edges of blocks of 16 rows and columns, sums that end inside a batch. The bound
    is that of the lists above; the gate's sigmoid (at most 1, slope 1/4) adds a few roundings of the result."""
    ops = hip_ops.HipOps("cuda:0", torch.bfloat16)
    assert ops._lazy("experts").cdll.tis_grouped_split(0, heads, rows, c_long(rows), N, K)
    g = torch.Generator().manual_seed(N + rows)
    x, w = torch.randn(rows, heads * K, generator=g).bfloat16(), (torch.randn(heads, N, K, generator=g) * K ** -0.5).bfloat16()
    gate = torch.randn(rows, heads * N + 3, generator=g)
    per_head = x.double().view(rows, heads, K)
    want = torch.einsum("rhk,hnk->rhn", per_head, w.double())
    size = torch.einsum("rhk,hnk->rhn", per_head.abs(), w.double().abs())
    for gated in (False, True):
        out = torch.full((rows, 2 + heads * (N + 3)), 7.0, device="cuda")
        ops.heads_linear(x.cuda(), w.cuda(), out, N + 3, 2, gate=gate.cuda()[:, 3:] if gated else None)
        got = out[:, 2:].reshape(rows, heads, N + 3).double().cpu()
        assert (got[..., N:] == 7.0).all() and (out[:, :2] == 7.0).all()
        factor = torch.sigmoid(gate[:, 3:].double()).view(rows, heads, N) if gated else 1.0
        assert ((got[..., :N] - want * factor).abs() <= size * (K / 4) * 2.0 ** -24 + want.abs() * 2.0 ** -20).all()
