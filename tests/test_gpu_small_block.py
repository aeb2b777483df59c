"""A small 32-bit block in one kernel against the separate kernels."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from tiny_inference_server_amd.ops import hip_ops

pytestmark = pytest.mark.gpu

# width, heads, kv heads, head size, hidden, page size
SIZES = [(64, 8, 2, 8, 176, 16), (64, 2, 1, 32, 192, 16), (48, 12, 3, 4, 64, 8), (20, 2, 1, 4, 12, 4), (4, 1, 1, 40, 4, 16), (32, 10, 5, 4, 100, 1),
         (60, 5, 1, 12, 188, 16), (40, 16, 8, 4, 8, 3), (36, 1, 1, 36, 68, 32)]


@pytest.mark.parametrize("D,H,G,HD,F,ps", SIZES)
@pytest.mark.parametrize("window,interleaved,rotary", [(0, False, True), (5, True, True), (0, False, False)])
def test_against_separate_kernels(D, H, G, HD, F, ps, window, interleaved, rotary):
    """Rows that see 1 key up to as many as the kernel takes, and a strided input; pages hold numbers that no row may see, infinities among them. Both sides
    are 32-bit sums of up to 512 terms in different orders, through two norms: 2e-6 of the largest value apart (a sum's error grows with the root of
    its terms, here some 23 roundings of 6e-8)."""
    ops = hip_ops.HipOps("cuda:0", torch.float32)
    gen = torch.Generator().manual_seed(D + window)

    def normal(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen) * std).cuda()

    taken = 0
    for lens in ([1, 2, 31, 33, 64, 65], [127, 1, 257], [512, 3, 1], [7]):
        M, keys = len(lens), max(lens)
        width = -(-keys // ps) + 1
        if not ops.small.cdll.tis_small_block_takes(M, D, F, H, G, HD, keys, ps):
            continue
        taken += 1
        plane = normal(M * width, 2, G, ps, HD)
        tables = torch.randperm(M * width, generator=gen).to(torch.int32).view(M, width)
        for i, n in enumerate(lens):                       # what a page holds beyond the request's keys is not read
            page, at = divmod(n - 1, ps)
            plane[int(tables[i, page]), 0].view(G, ps, HD)[:, at:] = float("inf")
            plane[int(tables[i, page]), 1].view(G, HD, ps)[:, :, at:] = float("nan")
            plane[tables[i, page + 1:].long()] = float("inf")
        seq = torch.randperm(M, generator=gen)
        pos = torch.tensor([lens[i] - 1 for i in seq], dtype=torch.int32)
        slots = torch.tensor([int(tables[i, (lens[i] - 1) // ps]) * ps + (lens[i] - 1) % ps for i in seq], dtype=torch.int32)
        batch = SimpleNamespace(positions=pos.cuda(), row_seq=seq.to(torch.int32).cuda(), write_slots={"g": slots.cuda()}, block_tables={"g": tables.cuda()},
                                max_kv_len=keys, max_seq_rows=1, n_rows=M, extras={}, seq_rows=[])
        x = normal(M, D + 4)[:, :D]
        gains = [1.0 + normal(D, std=0.1) for _ in range(2)]
        w_qkv, w_o = normal((H + 2 * G) * HD, D, std=D ** -0.5), normal(D, H * HD, std=(H * HD) ** -0.5)
        w_gu, w_down = normal(2 * F, D, std=D ** -0.5), normal(D, F, std=F ** -0.5)
        angles = torch.rand(keys, HD // 2, generator=gen).double() * 6.28
        table = torch.stack((torch.cos(angles), torch.sin(angles)), -1).float().cuda() if rotary else None
        scale = HD ** -0.5

        apart = plane.clone()
        q = ops.qkv_rope(x, w_qkv, (gains[0], 1e-5), batch.positions, batch.write_slots["g"], table, apart, H, G, HD, ps, interleaved)
        att = ops.paged_attention(q, apart, batch, "g", H, G, HD, window, scale)
        mid = ops.linear(att, w_o, residual=x)
        want = ops.linear(ops.linear_swiglu(mid, w_gu, rms=(gains[1], 1e-6)), w_down, residual=mid)

        got = ops.small_block(x, batch, "g", plane, ((gains[0], 1e-5), (gains[1], 1e-6)), (w_qkv, w_o, table, interleaved, H, G, HD, window, scale), (w_gu, w_down))
        assert float((got - want).abs().max() / want.abs().max()) < 2e-6
        # the cache: the same but for the rows' own slots, and those but for the order of sums
        torch.testing.assert_close(plane, apart, rtol=2e-6, atol=2e-6, equal_nan=True)
        own = torch.zeros(plane.shape[0], ps, dtype=torch.bool, device="cuda")
        own.view(-1)[slots.long()] = True
        for side, there in ((0, own[:, None, :, None]), (1, own[:, None, None, :])):
            shape = (-1, G, ps, HD) if side == 0 else (-1, G, HD, ps)
            a, b = (t[:, side].reshape(shape).nan_to_num(7.0, 8.0) for t in (plane, apart))
            assert torch.equal(a.masked_fill(there, 0), b.masked_fill(there, 0))
    assert taken >= 2


def test_what_it_leaves_alone():
    """Steps that bring a request several rows, blocks beyond a compute unit and rows that see more keys go to the separate kernels; the entry point refuses them."""
    ops = hip_ops.HipOps("cuda:0", torch.float32)
    takes = ops.small.cdll.tis_small_block_takes
    assert takes(512, 64, 176, 8, 2, 8, 512, 16) and not takes(3, 64, 176, 8, 2, 8, 513, 16) and not takes(513, 64, 176, 8, 2, 8, 512, 16)
    assert not takes(3, 128, 176, 8, 2, 8, 64, 16) and not takes(3, 64, 176, 8, 3, 8, 64, 16) and not takes(3, 64, 174, 8, 2, 8, 64, 16)
    assert not takes(3, 64, 196, 8, 2, 8, 64, 16) and not takes(3, 64, 176, 16, 2, 8, 64, 16) and not takes(3, 64, 176, 8, 8, 8, 64, 16)
    assert ops.small_block(None, SimpleNamespace(max_seq_rows=2, n_rows=2), "g", None, None, None, None) is None
    p = hip_ops._ptr(torch.zeros(64, device="cuda"))
    with pytest.raises(hip_ops.KernelError):
        ops.small.tis_small_block(p, 64, p, 64, p, 0.0, p, p, p, 0.0, p, p, hip_ops._ptr(None), 0, p, p, p, p, 1, p, 1, 128, 176, 8, 2, 8, 16, 0, 1.0, 16, ops._stream())


def test_a_small_call_leaves_a_larger_one_its_lds():
    """The kernel's limit of dynamic LDS is the process's: a call that needs little must not lower it under one that another thread is about to launch."""
    ops = hip_ops.HipOps("cuda:0", torch.float32)
    D, H, G, HD, F, ps, keys = 64, 8, 2, 8, 176, 16, 16
    batch = SimpleNamespace(positions=torch.tensor([keys - 1], dtype=torch.int32).cuda(), row_seq=torch.zeros(1, dtype=torch.int32).cuda(),
                            write_slots={"g": torch.tensor([keys - 1], dtype=torch.int32).cuda()}, block_tables={"g": torch.zeros(1, 1, dtype=torch.int32).cuda()},
                            max_kv_len=keys, max_seq_rows=1, n_rows=1, extras={}, seq_rows=[])

    def ones(*shape):
        return torch.ones(*shape, device="cuda")

    norm = (ones(D), 1e-5)
    y = ops.small_block(ones(1, D), batch, "g", ones(1, 2, G, ps, HD), (norm, norm),
                        (ones((H + 2 * G) * HD, D), ones(D, H * HD), None, False, H, G, HD, 0, 1.0), (ones(2 * F, D), ones(D, F)))
    torch.cuda.synchronize()
    assert y is not None and ops.small.cdll.tis_small_block_lds() == 160 * 1024
