"""Products of a model's own layers: at the row counts of prompts every tile of the tiled product, the gate taken on its sums, and the
choice between it and the library's product; in 32 bits the norm and the gate inside the product of few rows."""
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


@pytest.mark.parametrize("M", [129, 300, 1024, 1025, 2048, 2049])
def test_products_by_rows(ops, M):
    """Widths of the library's list and another: up to the limit the tiles, beyond it what linear takes. The same sums in the same order
    either way, so the same bits; a residual whose rows the library does not take, too."""
    for i, (N, K) in enumerate(((2304, 1536), (1536, 4096), (1000, 640))):
        x, w, res = rnd((M, K), 10 + i).cuda(), rnd((N, K), 20 + i, K ** -0.5).cuda(), rnd((M, N + 8), 30 + i).cuda()[:, 4:N + 4]
        gain = (1 + 0.1 * torch.randn(K, generator=torch.Generator().manual_seed(5))).cuda()
        want = x.double() @ w.double().t()
        torch.testing.assert_close(ops.linear_by_rows(x, w, residual=res).double(), want + res.double(), rtol=2e-2, atol=2e-2)
        whole = res.contiguous()
        if M <= 1024:                   # on the tiles either way
            assert torch.equal(ops.linear_by_rows(x, w, residual=res), ops.linear_by_rows(x, w, residual=whole))
        assert torch.equal(ops.linear_by_rows(x, w, residual=whole), ops.linear(x, w, residual=whole))
        assert torch.equal(ops.linear_by_rows(x, w, rms=(gain, 1e-5)), ops.linear(x, w, rms=(gain, 1e-5)))
        assert torch.equal(ops.linear_swiglu(x, w, rms=(gain, 1e-5)), ops.swiglu(ops.linear(x, w, rms=(gain, 1e-5))))


@pytest.mark.parametrize("M", [129, 257, 640, 1531, 2048])
def test_library_and_tiles_give_the_same_bits(ops, M):
    """At every width of the library's list: which of the two a layer's product takes is not seen in its result."""
    for i, (N, K) in enumerate(sorted(ops.library_widths)):
        x, w, res = ops.empty(M, K), rnd((N, K), 60 + i, K ** -0.5).cuda(), rnd((M, N), 80 + i).cuda()
        x.copy_(rnd((M, K), 70 + i))
        for residual in (None, res):
            tiles = ops._linear_tiles(x, w, residual, ops.empty(M, N), N, 0, 0)
            assert torch.equal(ops._linear_library(x, w, residual), tiles), (N, K)


@pytest.mark.parametrize("tile,rows,N,K", [(6, 600, 1020, 1416), (7, 1531, 2044, 1992), (8, 900, 2044, 712), (1, 129, 2052, 648), (2, 600, 2044, 1416)])
@pytest.mark.parametrize("gated", [False, True])
def test_grouped_product_of_many_steps(ops, tile, rows, N, K, gated):
    """Eight groups of uneven sizes (one empty, one of a single entry) in the tiles that many steps of K bring: every entry the sum that
    the group's matrix gives, one whole row of a tile behind the other; the gate one rounding to bfloat16 further."""
    from ctypes import c_long
    lib = ops._lazy("experts")
    assert lib.cdll.tis_grouped_tile(1, 8, rows, c_long(2 * rows), N, K, 0) == tile
    x, w = rnd((rows, K), 41).cuda(), rnd((8, N, K), 42, K ** -0.5).cuda()
    order = torch.randperm(2 * rows, generator=torch.Generator().manual_seed(6))
    left = 2 * rows - 1
    sizes = [1, 0] + [left // 6 + d for d in (-30, 30, -3, 3, -1)]
    sizes.append(2 * rows - sum(sizes))
    lists = torch.zeros(8, rows, dtype=torch.int32)
    at, group_of = 0, torch.empty(2 * rows, dtype=torch.long)
    for e, n in enumerate(sizes):
        mine = order[at:at + n].sort().values
        lists[e, :n], group_of[mine], at = mine.to(torch.int32), e, at + n
    lists, counts = lists.cuda(), torch.tensor(sizes, dtype=torch.int32, device="cuda")
    out = torch.empty(2 * rows, N // 2 if gated else N, device="cuda", dtype=torch.bfloat16 if gated else torch.float32)
    ops._grouped(x, x.stride(0), 0, 2, w, out, out.shape[1], 0, lists, counts, rows, rows, act=2 if gated else 0, limit=7.0)
    for e in range(8):
        mine = (group_of == e).nonzero()[:, 0].cuda()
        want = x[mine // 2].double() @ w[e].double().t()
        if gated:
            g, u = want[:, 0::2].clamp(max=7.0), want[:, 1::2].clamp(-7.0, 7.0)
            torch.testing.assert_close(out[mine].double(), g * torch.sigmoid(1.702 * g) * (u + 1.0), rtol=8e-3, atol=2e-3)
        else:
            torch.testing.assert_close(out[mine].double(), want, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("tile,M,N,K", [(8, 1100, 2044, 2312), (8, 1281, 1536, 4096), (8, 2047, 1532, 4040), (9, 1433, 2052, 4104), (9, 1532, 2048, 5632)])
def test_tiles_of_96(ops, tile, M, N, K):
    """128 x 96 and 96 x 128, whole tiles and parts of one in both directions and in the steps: against exact sums, as every tile, and with the library's bits
    where it has the width."""
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
    if (N, K) in ops.library_widths:
        assert torch.equal(out[:M], ops.linear(x, w, res, None, None, False, "library"))


@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (3, 352, 64), (16, 30, 4), (17, 352, 176), (70, 98, 260), (16, 2000, 1024), (33, 20, 1020)])
def test_norm_and_gate_inside_the_32_bit_product(M, N, K):
    """The same bits as the norm's, the product's and the gate's own kernels one after the other, on strided rows too; beyond the widths that
    fuse, the separate kernels."""
    ops = hip_ops.HipOps("cuda:0", torch.float32)
    g = torch.Generator().manual_seed(M + N + K)
    x = (torch.randn(M, K + 8, generator=g) * 3).cuda()[:, 4:K + 4]
    w, res, gain = torch.randn(N, K, generator=g).cuda(), torch.randn(M, N, generator=g).cuda(), torch.randn(K, generator=g).cuda()
    rms = (gain, 1e-5)
    assert ops._plain_fuses(x, w, rms) and not ops._plain_fuses(x[:, 1:], w, rms)
    normed = ops.rmsnorm(x, *rms)
    assert torch.equal(ops.linear(x, w, rms=rms), ops.linear(normed, w))
    assert torch.equal(ops.linear(x, w, rms=rms, residual=res), ops.linear(normed, w, residual=res))
    assert torch.equal(ops.linear_swiglu(x, w, rms=rms), ops.swiglu(ops.linear(normed, w)))
    assert torch.equal(ops.linear_swiglu(x, w), ops.swiglu(ops.linear(x.contiguous(), w)))
    assert not ops.gemm_plain.cdll.tis_gemm_plain_fuses(M, N, 1028)


@pytest.mark.parametrize("M,N,K,inside", [(3, 352, 64, True), (16, 4096, 128, True), (33, 1024, 100, True), (17, 2064, 128, False), (5, 352, 132, False), (70, 98, 260, False),
                                          (33, 20, 1020, False)])
def test_when_the_norm_goes_inside_the_32_bit_product(M, N, K, inside):
    """Up to 128 inner columns and 256 tiles, launched and in a graph. The same bits each way."""
    ops = hip_ops.HipOps("cuda:0", torch.float32)
    g = torch.Generator().manual_seed(M + N + K)
    x, w, gain = (torch.randn(M, K, generator=g) * 3).cuda(), torch.randn(N, K, generator=g).cuda(), torch.randn(K, generator=g).cuda()
    rms, norms, inner = (gain, 1e-5), [], ops.rmsnorm
    normed = inner(x, *rms)
    want = ops.linear(normed, w), ops.swiglu(ops.linear(normed, w))
    ops.rmsnorm = lambda *a, **k: (norms.append(1), inner(*a, **k))[1]
    both = lambda: (ops.linear(x, w, rms=rms), ops.linear_swiglu(x, w, rms=rms))
    assert all(torch.equal(a, b) for a, b in zip(both(), want)) and len(norms) == (0 if inside else 2)
    norms.clear()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = both()
    for _ in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want))
    assert len(norms) == (0 if inside else 2)


@pytest.mark.parametrize("groups,rows,top,N,K", [(64, 40, 2, 96, 1024), (70, 127, 2, 520, 136), (33, 17, 3, 64, 2048), (2, 23, 2, 132, 40), (130, 100, 1, 48, 264)])
def test_few_entries_in_many_groups(ops, groups, rows, top, N, K):
    """The product straight from memory with lists of up to several tiles of 16 entries: groups without an entry, of one, and the first of many;
    the sums against 64 bits, lines that no list names left alone."""
    from ctypes import c_long
    lib = ops._lazy("experts")
    assert lib.cdll.tis_grouped_tile(1, groups, rows, c_long(rows * top), N, K, 0) == -1
    g = torch.Generator().manual_seed(groups + rows)
    x, w = rnd((rows, K), 51).cuda(), rnd((groups, N, K), 52, K ** -0.5).cuda()
    lists, counts = torch.zeros(groups, rows, dtype=torch.int32), [0] * groups
    group_of = torch.full((rows * top,), -1)
    for e in range(rows * top):
        if e == 5:
            continue                                     # an entry of nobody
        to = 0 if e % top == 0 and rows > 20 else int(torch.randint(0, groups, (1,), generator=g))
        if counts[to] < rows:
            lists[to, counts[to]], group_of[e] = e, to
            counts[to] += 1
    out = torch.full((rows * top, N), 7.0, device="cuda")
    ops._grouped(x, x.stride(0), 0, top, w, out, N, 0, lists.cuda(), torch.tensor(counts, dtype=torch.int32, device="cuda"), rows, rows)
    for e in range(rows * top):
        if group_of[e] < 0:
            assert bool((out[e] == 7.0).all())
        else:
            torch.testing.assert_close(out[e].double(), w[group_of[e]].double() @ x[e // top].double(), rtol=1e-4, atol=1e-4)


# rows, heads, key/value heads, head size, inner columns, page size, the tile that the product takes
@pytest.mark.parametrize("M,H,G,HD,K,ps,tile", [
    (2048, 12, 3, 128, 1536, 16, 2), (1101, 12, 3, 128, 1536, 16, 8), (500, 12, 3, 128, 1032, 16, 5), (300, 12, 2, 64, 520, 16, 7), (700, 30, 1, 128, 1032, 32, 4),
    (2044, 56, 4, 128, 1544, 16, 0), (1020, 44, 2, 128, 1032, 16, 1), (2049, 49, 1, 96, 264, 48, 3), (333, 6, 1, 256, 520, 16, 6), (1433, 12, 2, 128, 4104, 16, 9)])
def test_queries_keys_and_values_from_the_product(ops, monkeypatch, M, H, G, HD, K, ps, tile):
    """Turned and cached by the product against the product, then the rotary kernel: the same bits in the queries and in every slot of the cache that a row writes,
    and nothing in the others; with every tile, heads that begin inside tiles, and keys and values that are not kept."""
    assert ops.gemm_tiles.cdll.tis_gemm_tiles_pick(M, (H + 2 * G) * HD, K) == tile
    gen = torch.Generator().manual_seed(M)
    x, w = rnd((M, K), 1).cuda(), rnd(((H + 2 * G) * HD, K), 2, K ** -0.5).cuda()
    gain = (1 + 0.1 * torch.randn(K, generator=gen)).cuda()
    pages = M // ps + 3
    pos = torch.randint(0, 4000, (M,), generator=gen).to(torch.int32).cuda()
    slots = torch.arange(5, 5 + M, dtype=torch.int32)             # consecutive, as a portion's are, but for some that change places
    swap = torch.randperm(M, generator=gen)[:40]
    slots[swap] = slots[swap.flip(0)]
    slots = slots.cuda()
    angle = torch.arange(4000)[:, None] * torch.rand(HD // 2, generator=gen)
    table = torch.stack((angle.cos(), angle.sin()), -1).contiguous().cuda()
    monkeypatch.setattr(ops, "_layer_route", lambda *a, **k: "tiles")
    for write in (True, False):
        planes = [torch.full((pages, 2, G, ps, HD), 5.0, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        q = ops.qkv_rope(x, w, (gain, 1e-5), pos, slots, table, planes[0], H, G, HD, ps, write_cache=write)
        qkv = ops.linear(x, w, None, None, (gain, 1e-5), False, "tiles")
        want = ops.empty(M, H * HD)
        ops.rope_write_kv(qkv, pos, slots, table, planes[1], H, G, HD, ps, False, write, paired=True, q_out=want)
        assert torch.equal(q, want) and torch.equal(*planes) and bool((planes[0] != 5.0).any()) == write
