"""Small kernels that wait for memory more than they work: attention of the general kernel, the arg-max, and the arrays that a captured step
takes from the host by itself."""
from __future__ import annotations

import pytest
import torch

from tiny_inference_server_amd.ops import hip_ops
from tiny_inference_server_amd.ops.hip_ops import _ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("HD,offset", [(8, 0), (8, 2), (10, 0), (36, 0), (96, 0), (128, 0), (256, 0)])
def test_general_attention(HD, offset, dtype):
    """Rows that see 1 key up to more than a chunk of them, with a window and with slopes; head sizes that are whole pieces of 16 bytes, that
    are not, and keys that do not start on 16 bytes (`offset`). Pages hold numbers that no row may see. 32-bit sums of up to 1,100 terms lie
    1e-6 off; a result in bfloat16 is rounded once (2^-9)."""
    ops = hip_ops.HipOps("cuda:0", dtype)
    H, G, ps, lens = 4, 2, 16, [1, 2, 31, 33, 127, 130, 1024, 1090]
    gen = torch.Generator().manual_seed(HD)
    width = -(-max(lens) // ps)
    pages = width * len(lens)
    tables = torch.randperm(pages, generator=gen).to(torch.int32).view(len(lens), width)
    numbers = torch.randn(pages * 2 * G * ps * HD + offset, generator=gen).to(dtype)
    plane = numbers[offset:].view(pages, 2, G, ps * HD)
    q = torch.randn(len(lens), H * HD, generator=gen).to(dtype)
    slopes = torch.tensor([0.5, 0.25, 0.1, 0.01])
    for window, bias in ((0, None), (40, slopes)):
        want = torch.empty(len(lens), H, HD, dtype=torch.float64)
        for r, n in enumerate(lens):
            first = max(0, n - window) if window else 0
            keys = plane[tables[r].long(), 0].double().view(width, G, ps, HD).transpose(1, 2).reshape(-1, G, HD)[first:n]
            vals = plane[tables[r].long(), 1].double().view(width, G, HD, ps).permute(0, 3, 1, 2).reshape(-1, G, HD)[first:n]
            for h in range(H):
                s = keys[:, h // (H // G)] @ q[r, h * HD:(h + 1) * HD].double() * HD ** -0.5
                if bias is not None:
                    s = s + bias[h].double() * (torch.arange(first, n) - (n - 1))
                want[r, h] = torch.softmax(s, 0) @ vals[:, h // (H // G)]
        out = torch.empty(len(lens), H * HD, dtype=dtype, device="cuda")
        gpu = [t.cuda() for t in (q, numbers, tables, torch.arange(len(lens), dtype=torch.int32), torch.tensor([n - 1 for n in lens], dtype=torch.int32))]
        d_bias = None if bias is None else bias.cuda()
        ops.attn_generic.tis_attention_generic(ops.code, _ptr(gpu[0]), H * HD, _ptr(gpu[1][offset:]), _ptr(gpu[2]), width, _ptr(gpu[3]), _ptr(gpu[4]),
                                                    _ptr(out), H * HD, len(lens), H, G, HD, ps, window, HD ** -0.5, _ptr(d_bias), ops._stream())
        t = 4e-6 if dtype == torch.float32 else 2.0 ** -8
        torch.testing.assert_close(out.cpu().double().view_as(want), want, rtol=t, atol=t)


@pytest.mark.parametrize("V", [1, 3, 64, 1023, 4099, 24576, 24580, 24583, 48000, 100001])
def test_argmax(V):
    """The first of the largest values, wherever they lie: one row each for the ends of a thread's pieces and for ties; a row of -inf, whose first is the
    row's first, wherever the row begins."""
    ops = hip_ops.HipOps("cuda:0", torch.float32)
    x = torch.randn(10, V, generator=torch.Generator().manual_seed(V)).clamp(max=2.0)       # (many ties at 2)
    for r, at in enumerate((0, V - 1, V // 2, min(V - 1, 4095), min(V - 1, 24575), min(V - 1, 24576))):
        x[r, at] = 9.0
    x[8, V // 3:] = 3.0
    x[9] = -float("inf")
    for shift in (0, 1):                                   # rows that start on 16 bytes, and rows that do not
        rows = torch.zeros(10, -(-V // 4) * 4 + 4 + shift, device="cuda")[:, shift:V + shift]
        rows.copy_(x)
        assert ops.argmax(rows).cpu().tolist() == x.argmax(-1).tolist()


@pytest.mark.parametrize("ints", [4, 2044, 2048, 2052, 16384, 40004])
def test_a_captured_step_takes_its_arrays_from_the_host(ints):
    """Replays take the two sets in turn, with other work between them, two of them launched before either is waited for; the GPU says how many have been taken."""
    ops = hip_ops.HipOps("cuda:0", torch.bfloat16)
    n = ops.upload_counters(ints)
    assert n == min(8, max(1, -(-ints // 2048)))
    ring = torch.zeros(2, ints, dtype=torch.int32, pin_memory=True)
    sent, done = torch.zeros(n, dtype=torch.int32, device="cuda"), torch.zeros(n, dtype=torch.int32, pin_memory=True)
    out, seen = torch.zeros(ints, dtype=torch.int32, device="cuda"), torch.zeros(ints, dtype=torch.int32, device="cuda")
    ops.upload_ring(ring, out, sent, done)               # (launched, then captured: the counters go on)
    torch.cuda.synchronize()
    assert done.tolist() == [1] * n
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.upload_ring(ring, out, sent, done)
        torch.add(out, 0, out=seen)
    for k in range(1, 12, 2):
        want = [torch.arange(ints, dtype=torch.int32) * (k + u) + 7 * u for u in (0, 1)]
        got = []
        for u in (0, 1):
            ring[(k + u) % 2].copy_(want[u])
            graph.replay()
            got.append(seen.clone())
        torch.cuda.synchronize()
        assert done.tolist() == [k + 2] * n
        for a, b in zip(got, want):
            assert torch.equal(a.cpu(), b)
    with pytest.raises(hip_ops.KernelError):
        ops.upload_ring(ring[:, :-2], out, sent, done)
