"""The parts that attention's tiles are cut into, as the host lists them for the tile kernel."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from tiny_inference_server_amd.ops import hip_ops
from tiny_inference_server_amd.ops.hip_ops import _ptr, attention_items, attention_launch_plan, first_key, tile_columns, tile_pieces

# (position, rows) per request
STEPS = {"one": [(0, 2048)], "odd": [(0, 1), (0, 1531), (7, 0), (3000, 333), (0, 64), (129, 17)], "late": [(4001, 700)], "short": [(0, 33), (31, 16)],
         "many": [(i * 37, 100 + 61 * i) for i in range(9)], "deep": [(8000, 40), (12, 1)]}


def rows_of(step):
    firsts = np.cumsum([0] + [n for _, n in step])
    return [(int(firsts[i]), p0, n) for i, (p0, n) in enumerate(step)]


@pytest.mark.parametrize("window", [0, 1, 100, 1024, -512, -64])
@pytest.mark.parametrize("splits,most", [(1, 1 << 20), (2, 30), (3, 22), (8, 8), (4, 1)])
@pytest.mark.parametrize("step", sorted(STEPS))
def test_every_part_of_every_tile_once(step, splits, most, window):
    """Tile by tile with the kernel's own arithmetic: how many parts it has and how long each is; longest first."""
    seq_rows = rows_of(STEPS[step])
    for group in (1, 4, 32):
        _, _, tiles, _ = attention_items(seq_rows, group, 32)
        got = tile_pieces(seq_rows, tiles, splits, most, window)
        want, chain = set(), {}
        for first, count in tiles.tolist():
            line = next(i for i, (f, _, n) in enumerate(seq_rows) if f <= first < f + n)
            pos = seq_rows[line][1] + first - seq_rows[line][0]
            k_lo = first_key(pos, window) & ~31
            steps = (pos + count - k_lo + 31) // 32
            parts = max(1, min(splits, (steps + most - 1) // most))
            per = (steps + parts - 1) // parts
            for s in range(parts):
                want.add((first, count + 256 * s, pos, line))
                chain[(first, s)] = min(steps, s * per + per) - s * per
        assert {tuple(e) for e in got.tolist()} == want and len(got) == len(want) and got.dtype == np.int32
        lengths = [chain[(f, c >> 8)] for f, c, _, _ in got.tolist()]
        assert lengths == sorted(lengths, reverse=True)


@pytest.mark.parametrize("tile_cols", [0, 32])
@pytest.mark.parametrize("group", [1, 3, 4, 16, 32, 48, 100])
def test_one_prompt_is_cut_like_a_prompt_among_others(group, tile_cols):
    """A request alone in its step, against the same beside one without rows, whose lists are made over all requests."""
    for m in (2, 3, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 1000, 1531, 2048, 6143, 6144, 6145):
        for f, p0 in ((0, 0), (5, 1), (0, 31), (7, 4001)):
            if group > 32 and tile_cols:        # (the tile kernel takes no such groups)
                continue
            alone, among = (attention_items(rows, group, tile_cols, 3) for rows in ([(f, p0, m)], [(f, p0, m), (f + m, 9, 0)]))
            assert alone[0] == among[0] and alone[3] == among[3]
            assert all(np.array_equal(x, y) and x.dtype == y.dtype for x, y in zip(alone[1:3], among[1:3]))


def test_a_tile_of_no_request_is_refused():
    with pytest.raises(hip_ops.KernelError, match="no request's"):
        tile_pieces([(4, 0, 0), (8, 0, 32)], np.array([[4, 32]], dtype=np.int32), 2, 8)


@pytest.mark.parametrize("total", [1, 255, 256, 257, 300, 511, 512, 513, 1000])
@pytest.mark.parametrize("dim,two", [(128, True), (256, False)])
def test_the_grid_takes_every_piece_once(total, dim, two):
    """What the kernel makes of its workgroups: two a compute unit, or one where heads are wide."""
    units, lib = 256, hip_ops.library(f"attention_mfma@{dim}").cdll
    took = [lib.tis_attention_mfma_piece_of(i, total, units) for i in range(total)]
    assert sorted(took) == list(range(total))
    if not two:
        assert took == list(range(total))
        return
    beside = [(took[i], took[i + units]) for i in range(min(units, max(0, total - units)))]
    assert all(b == min(2 * units, total) - 1 - a for a, b in beside)        # the longest has the shortest beside it


@pytest.mark.gpu
@pytest.mark.parametrize("dim,H,G,window,sink,page", [(128, 12, 3, 0, 0, 16), (128, 16, 4, 700, 0, 16), (64, 8, 8, -512, 0, 16), (256, 8, 2, 0, 1, 32), (48, 32, 1, 0, 0, 48)])
@pytest.mark.parametrize("step", sorted(STEPS))
def test_listed_parts_give_the_same_bits(dim, H, G, window, sink, page, step):
    """The list's flat grid, and the flat grid of tiles that are not cut, against the grid of tiles, heads and splits, which the first entry points of
    the library launch: the same bits."""
    ops = hip_ops.HipOps("cuda:0", torch.bfloat16)
    seq_rows, group = rows_of(STEPS[step]), H // G
    n, gen = sum(r[2] for r in seq_rows), torch.Generator().manual_seed(dim)
    nb, items, tiles, steps = attention_items(seq_rows, group, tile_columns(dim))
    width = max(-(-(p0 + m) // page) for _, p0, m in seq_rows)
    tables = torch.randperm(width * len(seq_rows), generator=gen).to(torch.int32).view(len(seq_rows), width).cuda()
    plane = torch.randn(width * len(seq_rows), 2 * G * page * dim, generator=gen).to(torch.bfloat16).cuda()
    q = torch.randn(n, H * dim, generator=gen).to(torch.bfloat16).cuda()
    seq = torch.tensor([i for i, (_, _, m) in enumerate(seq_rows) for _ in range(m)], dtype=torch.int32).cuda()
    pos = torch.tensor([p0 + k for _, p0, m in seq_rows for k in range(m)], dtype=torch.int32).cuda()
    lists = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (items, tiles)]
    lib = hip_ops.library(f"attention_mfma@{dim}")
    for cuts in ((1, 1 << 20), (3, 20), (8, 8)):
        lp = attention_launch_plan(n, len(items), len(tiles), steps, False, width * page, H, G, dim)
        stride = max(lp.n_splits, cuts[0])
        work = torch.empty(n * H * stride * (dim + 2) + n, device="cuda")
        ml, rs = work[n * H * stride * dim:], work[n * H * stride * (dim + 2):]
        outs = []
        for listed in (False, True):
            out = torch.full((n, H * dim), 9.0, dtype=torch.bfloat16, device="cuda")
            args = (_ptr(q), q.stride(0), _ptr(plane), _ptr(tables), width, _ptr(seq), _ptr(pos), _ptr(lists[0]) if len(items) else None, len(items), nb, _ptr(lists[1]), len(tiles),
                    _ptr(out), out.stride(0), _ptr(work), _ptr(ml), n, H, G, dim, page, window, dim ** -0.5, lp.n_splits, lp.min_steps, cuts[0], cuts[1], _ptr(rs), sink, None, None)
            if listed:
                pieces = tile_pieces(seq_rows, tiles, *cuts, window)
                on_gpu = torch.from_numpy(pieces).cuda()
                few = 2 if cuts[0] == 1 else ops.units      # (a chip so small that the tiles are more than its units)
                lib.tis_attention_mfma_pieces(*args, None, 0, 0.0, _ptr(on_gpu) if cuts[0] > 1 else None, len(pieces) if cuts[0] > 1 else 0, few, ops._stream())
            else:
                lib.tis_attention_mfma_sink(*args, ops._stream())
            torch.cuda.synchronize()
            outs.append(out)
        assert torch.equal(*outs) and bool(torch.isfinite(outs[0]).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dim,H,G,sink", [(128, 8, 2, 0), (64, 8, 8, 1), (48, 5, 1, 0), (256, 8, 2, 0)])
@pytest.mark.parametrize("cuts", [(2, 60), (4, 40), (5, 30), (9, 16), (80, 1)])
def test_merged_rows_do_not_depend_on_how_many_there_are(dim, H, G, sink, cuts):
    """Rows merged by four waves (few rows times heads) and by one (more): the same bits."""
    ops, page, window = hip_ops.HipOps("cuda:0", torch.bfloat16), 16, 0
    gen, p0, m = torch.Generator().manual_seed(dim), 2600, 100
    q1 = torch.randn(m, H * dim, generator=gen).to(torch.bfloat16).cuda()
    width = -(-(p0 + m) // page)
    plane = torch.randn(width, 2 * G * page * dim, generator=gen).to(torch.bfloat16).cuda()
    lib, outs = hip_ops.library(f"attention_mfma@{dim}"), []
    for copies in (1, 2048 // (m * H) + 1, 8192 // (m * H)):
        seq_rows = [(i * m, p0, m) for i in range(copies)]
        n = m * copies
        assert n * H <= 2048 if copies == 1 else 2048 < n * H <= 8192
        nb, items, tiles, steps = attention_items(seq_rows, H // G, tile_columns(dim))
        assert not len(items)
        q, tables = q1.repeat(copies, 1), torch.arange(width, dtype=torch.int32).repeat(copies, 1).cuda()
        seq = torch.arange(copies, dtype=torch.int32).repeat_interleave(m).cuda()
        pos = (torch.arange(m, dtype=torch.int32) + p0).repeat(copies).cuda()
        on_gpu = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (tiles, tile_pieces(seq_rows, tiles, *cuts, window))]
        work = torch.empty(n * H * cuts[0] * (dim + 2) + n, device="cuda")
        ml, rs = work[n * H * cuts[0] * dim:], work[n * H * cuts[0] * (dim + 2):]
        out = torch.full((n, H * dim), 9.0, dtype=torch.bfloat16, device="cuda")
        lib.tis_attention_mfma_pieces(
            _ptr(q), q.stride(0), _ptr(plane), _ptr(tables), width, _ptr(seq), _ptr(pos), None, 0, nb, _ptr(on_gpu[0]), len(tiles), _ptr(out), out.stride(0), _ptr(work),
            _ptr(ml), n, H, G, dim, page, window, dim ** -0.5, 1, 0, cuts[0], cuts[1], _ptr(rs), sink, None, None, None, 0, 0.0, _ptr(on_gpu[1]), len(on_gpu[1]), ops.units, ops._stream())
        torch.cuda.synchronize()
        outs.append(out)
    for out in outs[1:]:
        assert torch.equal(out, outs[0].repeat(len(out) // m, 1)) and bool(torch.isfinite(out).all())
