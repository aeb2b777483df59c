"""The Fesupel architecture on the GPU: each new kernel against plain torch, and the engine with its HIP kernels against
the plain implementation through every kind of schedule, in 32-bit and in bfloat16."""
import copy
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import fesupel_models as FM
import helpers as H
import plain_fesupel as pf
from test_gpu_fikevik import fake_batch
from torch_ops import TorchOps

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TOL = FM.TOL
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def hip_ops(dtype):
    from tiny_inference_server_amd.ops.hip_ops import HipOps
    return HipOps("cuda:0", DT[dtype])


def model(name, dtype="float32", seed=5):
    """In bfloat16 every expert is chosen (see fesupel_models.all_chosen); routing itself is tested in 32-bit and kernel
    by kernel in both types."""
    cfg = FM.CONFIGS[name] if dtype == "float32" else FM.all_chosen(FM.CONFIGS[name])
    w = FM.random_weights(cfg, seed)
    return copy.deepcopy(cfg), w, FM.as_f64(w)


def engine_for(cfg, w, dtype, **kw):
    from tiny_inference_server_amd.config import config_from_dict
    from tiny_inference_server_amd.engine import Engine
    kw.setdefault("max_requests", 4)
    kw.setdefault("page_size", 16)
    kw.setdefault("max_tokens", 1024)
    eng = Engine(config=config_from_dict(cfg), tensors=w, dtype=dtype, **kw)
    H.fill_cache_with_nan(eng)       # what a row may not see must not reach a result
    return eng


def close(a, b, dtype, what, tol=None):
    tol = tol or (2e-5 if dtype == "float32" else 1.6e-2)
    err = (a.float().cpu() - b.float().cpu()).abs().max().item()
    assert err <= tol * max(1.0, b.float().abs().max().item()), (what, err)


# ---- kernels ---------------------------------------------------------------------------------------------------

@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("Hq,G,kd,vd,chunk,cap", [(6, 2, 24, 40, 7, 3.0), (4, 4, 64, 16, 0, 0.0), (2, 1, 10, 200, 33, 30.0), (3, 1, 96, 48, 16, 1.0),
                                                  (16, 4, 32, 32, 5, 0.0), (1, 1, 64, 1, 1, 2.0), (5, 5, 7, 9, 300, 0.0)])
def test_attention_with_mixed_sigmoid_weights(dtype, Hq, G, kd, vd, chunk, cap):
    """Chunks that end mid-page, a whole prompt and a portion that goes on at 19 beside a new request; few rows, so
    the keys of a row are cut over several workgroups and added up."""
    ops, ref = hip_ops(dtype), TorchOps("cpu", DT[dtype])
    g = torch.Generator().manual_seed(kd + chunk)
    ps, n_pages = 8, 12
    tables = [[5, 2, 9, 0, 0, 0], [7, 1, 3, 11, 4, 0]]
    cols = Hq * kd + G * kd + G * vd + 3
    biases = [0.3 * torch.randn(s, generator=g) for s in (Hq * kd, G * kd, G * vd)]
    head_bias, talk = torch.randn(Hq, generator=g) - 1, torch.eye(Hq) + 0.4 * torch.randn(Hq, Hq, generator=g)
    planes = [torch.full((n_pages, G * ps * (kd + vd)), float("nan"), dtype=DT[dtype]) for _ in range(2)]
    planes[0] = planes[0].cuda()
    for seq_rows in ([(0, 0, 19)], [(0, 0, 21), (21, 19, 17)]):
        n = sum(r[2] for r in seq_rows)
        proj = torch.randn(n, cols, generator=g)
        slots = [0] if len(seq_rows) == 1 else [1, 0]
        tabs = [tables[1]] if len(seq_rows) == 1 else [tables[0], tables[1]]
        res = []
        for o, plane, dev in ((ops, planes[0], "cuda"), (ref, planes[1], "cpu")):
            b = fake_batch(seq_rows, slots, tabs, ps, dev)
            mv = lambda t: t.to(dev)
            q = o.attention_prepare(mv(proj)[:, 3:], 0, Hq * kd, Hq * kd + G * kd, b.positions, b.write_slots["g"], plane, Hq, G, kd, vd,
                                    ps, value_norm=False, q_bias=mv(biases[0]), k_bias=mv(biases[1]), v_bias=mv(biases[2]))
            res.append(o.mixed_sigmoid_attention(q, plane, b, "g", Hq, G, kd, vd, ps, chunk, 0.37, cap, mv(head_bias), mv(talk)))
        close(res[0], res[1], dtype, "attention")
        assert torch.isfinite(res[0].float()).all()


@pytest.mark.parametrize("Hq,G,kd,vd,chunk,cap", [(4, 1, 64, 64, 100, 30.0), (16, 4, 128, 128, 333, 0.0), (5, 5, 24, 32, 7, 2.0), (6, 2, 40, 16, 0, 0.0),
                                                  (2, 1, 128, 64, 64, 10.0), (13, 1, 16, 48, 1, 0.0), (8, 8, 32, 32, 1000, 5.0)])
def test_matrix_core_attention_with_mixed_sigmoid_weights(Hq, G, kd, vd, chunk, cap):
    """bfloat16 and pages of 16 slots: tiles of rows that cross chunk edges and page borders, a portion that goes on in the
    middle of a page beside a new request, and single rows whose keys are cut over many workgroups; the pool is full of
    NaN where nothing was written."""
    ops, ref = hip_ops("bfloat16"), TorchOps("cpu", torch.bfloat16)
    g = torch.Generator().manual_seed(kd + chunk)
    ps, n_pages = 16, 40
    perm = torch.randperm(n_pages, generator=g).tolist()
    tables = [perm[:18] + [0, 0], perm[18:38]]
    cols = Hq * kd + G * kd + G * vd
    head_bias, talk = torch.randn(Hq, generator=g) - 2, torch.eye(Hq) + 0.4 * torch.randn(Hq, Hq, generator=g)
    planes = [torch.full((n_pages, G * ps * (kd + vd)), float("nan"), dtype=torch.bfloat16) for _ in range(2)]
    planes[0] = planes[0].cuda()
    for seq_rows, slots, tabs in (([(0, 0, 203)], [0], [tables[1]]), ([(0, 0, 37), (37, 203, 70)], [1, 0], [tables[0], tables[1]]),
                                  ([(0, 37, 1), (1, 273, 1)], [1, 0], [tables[0], tables[1]]),
                                  ([(0, 38, 2), (2, 274, 1), (3, 0, 0)][:2], [1, 0], [tables[0], tables[1]])):
        n = sum(r[2] for r in seq_rows)
        proj = torch.randn(n, cols, generator=g)
        res = []
        for o, plane, dev in ((ops, planes[0], "cuda"), (ref, planes[1], "cpu")):
            b = fake_batch(seq_rows, slots, tabs, ps, dev)
            q = o.attention_prepare(proj.to(dev), 0, Hq * kd, Hq * kd + G * kd, b.positions, b.write_slots["g"], plane, Hq, G, kd, vd,
                                    ps, value_norm=False)
            res.append(o.mixed_sigmoid_attention(q, plane, b, "g", Hq, G, kd, vd, ps, chunk, kd ** -0.5, cap, head_bias.to(dev),
                                                 talk.to(dev)))
        assert ops._mixed_on_matrix_cores(res[0], kd, vd, ps, Hq)
        assert torch.isfinite(res[0].float()).all()
        close(res[0], res[1], "bfloat16", f"attention of {seq_rows}", tol=2.5e-2)


@pytest.mark.parametrize("heads,dim,resident", [(4, 128, 2), (16, 128, 1), (4, 64, 2), (16, 64, 1)])
def test_cuts_of_the_keys_for_what_a_unit_holds(heads, dim, resident):
    """The library tells how many workgroups a compute unit holds for its sizes, and the cuts that the kernel is called with fill two a unit
    where that many fit and one where one does (single rows: not one more); whatever the cuts, the same sums."""
    ops = hip_ops("bfloat16")
    assert min(2, ops._lazy(f"attention_mixed@{dim * 100000 + dim * 100 + -(-heads // 4)}").cdll.tis_attention_mixed_resident(heads)) == resident
    n, ps, G = 32, 16, max(1, heads // 4)
    g = torch.Generator().manual_seed(heads + dim)
    plane = (0.5 * torch.randn(64, G * ps * 2 * dim, generator=g)).to(torch.bfloat16).cuda()
    q = torch.randn(n, heads * dim, generator=g).to(torch.bfloat16).cuda()
    bias, talk = torch.full((heads,), -5.0).cuda(), (torch.eye(heads) + 0.2 * torch.randn(heads, heads, generator=g)).cuda()
    batch = fake_batch([(i, 600 + i, 1) for i in range(n)], list(range(n)), [torch.randperm(64, generator=g).tolist() for _ in range(n)], ps, "cuda")

    def parts():
        """The cuts, from how much of the work space a call writes."""
        ops._workspace.fill_(float("nan"))
        out = ops.mixed_sigmoid_attention(q, plane, batch, "g", heads, G, dim, dim, ps, 0, dim ** -0.5, 30.0, bias, talk)
        return int((~ops._workspace.isnan()).sum()) // (n * heads * dim), out

    cuts, out = parts()
    assert cuts == (16 if resident == 2 else 8) * ops.units // 256
    units, ops.units = ops.units, 1
    none, whole = parts()
    ops.units = units
    assert none == 0
    close(out, whole, "bfloat16", "sums of cuts", tol=1e-2)      # (one rounding to bfloat16 each, of sums in another order)


def test_mixed_weights_are_quotients_rounded_as_a_division_rounds_them():
    """The matrix-core kernel's weights, to the last bit: with scores of zero and biases that are whole numbers on base 2 a weight is
    1 / (1 + 2^n), the power is exact, and only the reciprocal rounds. Head 0's weight is a half; every other head takes its own weight
    less the rounded quotient times that half, so that what is left is the weight's error, exact in bfloat16. Half a unit of the last place
    is a division's error; the bound leaves the hundredth of one for a quotient next to the middle of two numbers."""
    ops = hip_ops("bfloat16")
    H, kd, vd, ps = 16, 128, 128, 16
    log2e = np.float32(1.4426950408889634)
    exponents = []
    for n in list(range(-23, 24)) + list(range(30, 60)) + [128, 300]:      # 1 + 2^n is exact, or 2^n to all 24 bits, or infinite: weight 0
        bias = np.float32(-n / float(log2e))
        for b in (bias, np.nextafter(bias, np.float32(np.inf)), np.nextafter(bias, np.float32(-np.inf))):
            if np.float32(-log2e * b) == n:
                exponents.append((n, float(b)))
                break
    assert len(exponents) >= 45
    plane = torch.zeros(1, ps * (kd + vd), dtype=torch.bfloat16)
    plane[0, ps * kd:] = 1.0
    for at in range(0, len(exponents), H - 1):
        part = exponents[at:at + H - 1]
        head_bias, talk, want = torch.zeros(H), torch.zeros(H, H), torch.full((H,), 0.5, dtype=torch.float64)
        talk[0, 0] = 1.0
        for h, (n, b) in enumerate(part, 1):
            want[h] = 1.0 / (1.0 + 2.0 ** n) if n < 128 else 0.0
            head_bias[h] = b
            talk[h, h], talk[h, 0] = 1.0, -2.0 * want[h].float()
        batch = fake_batch([(0, 0, 1)], [0], [[0]], ps, "cuda")
        out = ops.mixed_sigmoid_attention(torch.zeros(1, H * kd, dtype=torch.bfloat16, device="cuda"), plane.cuda(), batch, "g", H, 1, kd, vd, ps,
                                          0, 0.5, 0.0, head_bias.cuda(), talk.cuda()).double().cpu().view(H, vd)
        assert (out == out[:, :1]).all() and out[0, 0] == 0.5
        for h, (n, _) in enumerate(part, 1):
            weight = out[h, 0].item() + want[h].float().double().item()
            unit = float(np.spacing(np.float32(want[h].item()))) if want[h] > 0 else 0.0
            assert abs(weight - want[h].item()) <= 0.51 * unit, (n, weight, want[h].item(), (weight - want[h].item()) / (unit or 1.0))


def test_attention_of_many_rows_and_long_chunks():
    """Hundreds of rows (one workgroup a row, no key splits) over chunks longer than a block of keys."""
    ops, ref = hip_ops("float32"), TorchOps("cpu", torch.float32)
    g = torch.Generator().manual_seed(3)
    Hq, G, kd, vd, ps, n = 4, 2, 16, 8, 16, 700
    table = [list(torch.randperm(48, generator=g)[:44].tolist())]
    plane = torch.randn(48, G * ps * (kd + vd), generator=g)
    q = torch.randn(n, Hq * kd, generator=g)
    head_bias, talk = torch.randn(Hq, generator=g) - 3, torch.randn(Hq, Hq, generator=g)
    for chunk in (0, 300):
        outs = []
        for o, dev in ((ops, "cuda"), (ref, "cpu")):
            b = fake_batch([(0, 0, n)], [0], table, ps, dev)
            outs.append(o.mixed_sigmoid_attention(q.to(dev), plane.to(dev), b, "g", Hq, G, kd, vd, ps, chunk, 0.2, 4.0,
                                                  head_bias.to(dev), talk.to(dev)))
        close(outs[0], outs[1], "float32", f"chunks of {chunk}", tol=1e-4)


@pytest.mark.parametrize("Hh,G,D,V,K", [(4, 2, 12, 8, 4), (6, 3, 8, 4, 2), (2, 1, 20, 6, 1), (4, 2, 64, 32, 4), (2, 1, 128, 64, 3), (1, 1, 1, 8, 2),
                                        (3, 1, 6, 1, 1), (2, 2, 200, 20, 2), (2, 1, 33, 17, 3)])
def test_the_delta_rules_kernels(Hh, G, D, V, K):
    """The step before the walk and the walk: a whole prompt from an empty line, then portions and single rows that go on
    from used lines, beside a new request."""
    ops, ref = hip_ops("float32"), TorchOps("cpu", torch.float32)
    g = torch.Generator().manual_seed(D + V)
    C = 2 * G * D + Hh * V
    cols = 5 + C + Hh
    taps = torch.randn(C, K, generator=g) / K ** 0.5
    at = Hh * -(-V // 16) * D * 16           # the matrix state in blocks of 16 value channels, then the convolution's inputs
    floats = at + (K - 1) * C
    floats += -floats % 4 + 4                # lines start 16 bytes aligned
    states = [torch.zeros(3, floats), torch.zeros(3, floats).cuda()]
    for seq_rows, slots in (([(0, 0, 37)], [2]), ([(0, 37, 1), (1, 0, 9)], [2, 0]), ([(0, 9, 70), (70, 38, 2)], [0, 2]),
                            ([(0, 40, 1), (1, 79, 1)], [2, 0])):
        n = sum(r[2] for r in seq_rows)
        proj = torch.randn(n, cols, generator=g)
        decay = torch.rand(n, Hh * D, generator=g) * 0.5 + 0.5
        res = []
        for o, st, dev in ((ref, states[0], "cpu"), (ops, states[1], "cuda")):
            b = fake_batch(seq_rows, slots, None, 8, dev)
            u = o.delta_prepare(proj.to(dev), 5, 5 + C, taps.to(dev), st, at, b, Hh, G, D, V)
            o.conv_state_update(proj.to(dev), 5, C, K, st, at, b)
            res.append((u, o.delta_scan(u, 0, G * D, 2 * G * D, C, decay.to(dev), st, b, Hh, G, D, V)))
        close(res[1][0], res[0][0], "float32", "prepared rows", tol=1e-5)
        close(res[1][1], res[0][1], "float32", "outputs", tol=1e-4)
        close(states[1], states[0], "float32", "state lines", tol=1e-4)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,W", [(23, 44), (5, 328), (300, 1500)])
def test_row_kernels_of_the_block(dtype, n, W):
    from tiny_inference_server_amd.ops.hip_ops import ChosenExperts
    ops, ref = hip_ops(dtype), TorchOps("cpu", DT[dtype])
    g = torch.Generator().manual_seed(W)
    y0, y1 = torch.randn(n, W + 3, generator=g) * 3, torch.randn(n, W, generator=g) * 0.1
    g0, g1 = 1 + 0.3 * torch.randn(W, generator=g), 1 + 0.3 * torch.randn(W, generator=g)
    close(ops.normed_mean([(y0.cuda()[:, 3:], g0.cuda()), (y1.cuda(), g1.cuda())], 1e-5), ref.normed_mean([(y0[:, 3:], g0), (y1, g1)], 1e-5),
          "float32", "mean of two normed rows")
    close(ops.normed_mean([(y1.cuda(), g1.cuda())], 1e-6), ref.normed_mean([(y1, g1)], 1e-6), "float32", "one normed row")
    for act in ("relu2", "gelu_tanh", "silu", "sigmoid"):
        close(ops.activate_rows(y0.cuda()[:, 3:], act), ref.activate_rows(y0[:, 3:], act), dtype, act)
    z = torch.randn(n, 2 * 40 + 1, generator=g) * 2
    close(ops.gated_act(z.cuda(), 40, "clamped_swish", limit=0.8), ref.gated_act(z, 40, "clamped_swish", limit=0.8), dtype, "clamped gate")
    rank = 7
    low, w2, bias, rate = torch.randn(n, rank + 2, generator=g), torch.randn(W, rank, generator=g), torch.randn(W, generator=g), torch.rand(W // 4, generator=g)
    if W % 4 == 0:
        close(ops.lowrank_act(low.cuda()[:, 2:], w2.cuda(), bias.cuda(), "exp_softplus", rate=rate.cuda(), group=4),
              ref.lowrank_act(low[:, 2:], w2, bias, "exp_softplus", rate=rate, group=4), "float32", "decays")
    close(ops.lowrank_act(low.cuda()[:, 2:], w2.cuda(), None, "none"), ref.lowrank_act(low[:, 2:], w2, None, "none"), "float32", "low-rank product")
    # the residual sum with a row's chosen experts, identity experts, a gated shared term and a norm on the branch
    top, E = 3, 4
    x = torch.randn(n, W, generator=g)
    lines, extra, gate = torch.randn(n * top, W, generator=g), torch.randn(n, W, generator=g), torch.randn(n, 5, generator=g)
    ids = torch.randint(0, E + 2, (n, top), generator=g, dtype=torch.int32)
    wts = torch.rand(n, top, generator=g)
    rows = x.to(DT[dtype])
    res = []
    for o, dev in ((ops, "cuda"), (ref, "cpu")):
        ch = ChosenExperts(lines.to(dev), ids.to(dev), wts.to(dev), E, rows.to(dev), extra.to(dev), gate.to(dev)[:, 2:3])
        res.append(o.residual_norm(x.clone().to(dev), ch, y_rms=(g0.to(dev), 1e-5), copy=True, norm=("rms", g1.to(dev), None, 1e-5)))
    close(res[0][0], res[1][0], "float32", "sum", tol=1e-4 if dtype == "float32" else 2e-2)
    close(res[0][2], res[1][2], dtype, "the next norm", tol=1e-4 if dtype == "float32" else 3e-2)


@pytest.mark.parametrize("rank", [1, 15, 16, 17, 32, 33, 64, 65, 130, 257])
@pytest.mark.parametrize("n,C", [(1, 33), (257, 64), (299, 100), (513, 514), (90, 6000)])
def test_low_rank_projections_of_several_chunks_of_the_rank(rank, n, C):
    """The rank comes in chunks of 16, 32 or 64, rows by eight or (many rows times channels: the last two sizes) by 32 a workgroup: ranks of
    one chunk, of one more and of several, whole and not; the sums against 64 bits, the decays against the sums; and a row's bits do not
    depend on how many rows there are."""
    ops = hip_ops("float32")
    g = torch.Generator().manual_seed(rank * n + C)
    low, w2 = torch.randn(n, rank + 3, generator=g)[:, 1:1 + rank], torch.randn(C, rank, generator=g) * rank ** -0.5
    bias, rate = torch.randn(C, generator=g), torch.rand(C, generator=g) * 4
    on = lambda t: t.cuda()
    wide = torch.full((n, rank + 3), float("nan"))
    wide[:, 1:1 + rank] = low
    dev = on(wide)[:, 1:1 + rank]           # rows that begin beside a number that is none
    want = low.double() @ w2.double().T
    # `rank` products and as many additions, each within half a unit of the sum of magnitudes
    bound = (rank + 1) * 2.0 ** -24 * (low.double().abs() @ w2.double().abs().T)
    got = ops.lowrank_act(dev, on(w2), None, "none").cpu()
    assert ((got.double() - want).abs() <= bound).all()
    assert torch.equal(ops.lowrank_act(dev[n // 2:n // 2 + 1], on(w2), None, "none").cpu(), got[n // 2:n // 2 + 1])
    z = want + bias.double()
    close(ops.lowrank_act(dev, on(w2), on(bias), "exp_softplus", rate=on(rate), group=1),
          torch.exp(-rate.double() * torch.nn.functional.softplus(z)), "float32", "decays")
    close(ops.lowrank_decay(dev, on(w2), on(bias), 7.0), torch.exp(torch.nn.functional.logsigmoid(z) / 7.0), "float32", "decays of a sigmoid")


@pytest.mark.parametrize("rank", [4, 16, 20, 32, 64, 68, 132])
@pytest.mark.parametrize("n,C", [(1, 33), (257, 64), (513, 514), (90, 6000)])
def test_low_rank_projections_read_16_bytes_at_a_time(rank, n, C):
    """Rows that begin on 16 bytes, in steps of 16, beside a number that is none: the sums against 64 bits, and the bits of rows that begin
    in between, which are read one number at a time."""
    ops = hip_ops("float32")
    g = torch.Generator().manual_seed(rank * n + C)
    low, w2 = torch.randn(n, rank, generator=g), torch.randn(C, rank, generator=g) * rank ** -0.5
    bias, rate = torch.randn(C, generator=g).cuda(), (torch.rand(C, generator=g) * 4).cuda()

    def rows_at(column, columns):
        wide = torch.full((n, columns), float("nan"))
        wide[:, column:column + rank] = low
        return wide.cuda()[:, column:column + rank]
    aligned, between = rows_at(4, rank + 8), rows_at(1, rank + 3)
    assert aligned.data_ptr() % 16 == 0 and aligned.stride(0) % 4 == 0 and between.data_ptr() % 16
    w2 = w2.cuda()
    got = ops.lowrank_act(aligned, w2, None, "none")
    bound = (rank + 1) * 2.0 ** -24 * (low.double().abs() @ w2.cpu().double().abs().T)
    assert ((got.cpu().double() - low.double() @ w2.cpu().double().T).abs() <= bound).all()
    assert torch.equal(got, ops.lowrank_act(between, w2, None, "none"))
    assert torch.equal(ops.lowrank_act(aligned, w2, bias, "exp_softplus", rate=rate, group=1), ops.lowrank_act(between, w2, bias, "exp_softplus", rate=rate, group=1))
    assert torch.equal(ops.lowrank_decay(aligned, w2, bias, 7.0), ops.lowrank_decay(between, w2, bias, 7.0))


@pytest.mark.parametrize("n,N,top,groups", [(37, 8, 2, (4, 2)), (5, 12, 3, (3, 1)), (200, 16, 3, (2, 1)), (9, 6, 6, None), (64, 64, 4, (16, 3)),
                                            (33, 10, 1, (10, 1)), (20, 130, 5, (13, 2))])
def test_choice_in_groups(n, N, top, groups):
    ops, ref = hip_ops("float32"), TorchOps("cpu", torch.float32)
    g = torch.Generator().manual_seed(N)
    z, c = torch.randn(n, N + 2, generator=g) * 2, torch.randn(N, generator=g) * 0.1 - 0.5      # corrected scores are negative
    ids, w = ops.route_topk(z.cuda()[:, 2:], c.cuda(), 1.0, top, groups=groups, renorm=True)
    ids_r, w_r = ref.route_topk(z[:, 2:], c, 1.0, top, groups=groups, renorm=True)
    assert torch.equal(ids.cpu(), ids_r)
    close(w, w_r, "float32", "weights")
    assert torch.allclose(w.sum(-1).cpu(), torch.ones(n), atol=1e-5)
    if groups:
        per = N // groups[0]
        assert all(len({int(e) // per for e in row}) <= groups[1] for row in ids.cpu())


# ---- the engine ------------------------------------------------------------------------------------------------

@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(FM.CONFIGS))
def test_schedules(name, dtype):
    if name == "D" and dtype == "bfloat16":
        pytest.skip("the configuration of ones divides single numbers by their own size: bfloat16 rounding is all of it")
    cfg, w, w64 = model(name, dtype)
    key = (name, dtype)
    reqs = {f"r{i}": H.random_ids(cfg["vocab"], n, 40 + i) for i, n in enumerate([37, 1, 158, 23, 70])}
    eng = engine_for(cfg, w, dtype)
    tol = 3e-4 if name == "D" else None

    def check(got):
        if tol:
            assert FM.worst_error(key, cfg, w64, reqs, got)[0] <= tol
        else:
            FM.check(key, cfg, w64, reqs, got, dtype)

    for steps in (H.whole_trace(reqs), H.tail_decode_trace(reqs, tail=20), H.portions_trace(reqs, seed=3)):
        got = FM.run_trace(eng, steps)
        assert len(got) == sum(len(v) for v in reqs.values())
        check(got)
        eng.cache.check()
    steps, peak = H.mixed_trace(reqs, max_live=3, seed=4)
    eng = engine_for(cfg, w, dtype, max_requests=3, max_tokens=peak)
    check(FM.run_trace(eng, steps))
    eng.cache.check()


def needle_case(name, dtype, at, distance, side, chunk):
    cfg, w, _ = model(name, dtype)
    if chunk is not None:
        cfg["layers"][0]["mixer"]["left"]["mask"] = {"size": chunk}
    w = FM.sharpen(cfg, w, 3, 7, side)
    w64 = FM.as_f64(w)
    ids = [t if t not in (3, 7) else 11 for t in H.random_ids(cfg["vocab"], at + distance + 4, 60 + at)]
    ids[at], ids[at + distance] = 3, 7
    key = (name, dtype, "sharp", side, chunk)
    want = FM.plain_logits(key, cfg, w64, ids)
    without = list(ids)
    without[at] = 11
    moved = FM.relative_error(pf.forward(cfg, w64, without)[at + distance], want[at + distance])
    return key, cfg, w, w64, ids, want, moved


def run_three_ways(key, cfg, w, w64, ids, want, place, bound, dtype, tail=6):
    eng = engine_for(cfg, w, dtype)
    for steps in (H.whole_trace({"s": ids}), H.tail_decode_trace({"s": ids}, tail=tail), H.portions_trace({"s": ids}, sizes=(5, 2, 11))):
        got = FM.run_trace(eng, steps)
        err = FM.relative_error(got[("s", place)], want[place])
        assert err <= bound, (err, bound, place)
        FM.check(key, cfg, w64, {"s": ids}, got, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name,distance,side,chunk", [("A", 1, "left", None), ("C", 300, "left", 400), ("C", 150, "right", None),
                                                      ("B", 60, "right", None)])
def test_a_token_that_stands_out(name, distance, side, chunk, dtype):
    """A probe token that looks for a needle right before it or hundreds of tokens back, through attention's pages or the
    delta rule's state, with the needle on both sides of a page's border: whole, decoded alone, in portions."""
    for at in (15, 16):
        key, cfg, w, w64, ids, want, moved = needle_case(name, dtype, at, distance, side, chunk)
        assert moved >= 0.01, moved
        run_three_ways(key, cfg, w, w64, ids, want, at + distance, min(TOL[dtype], moved / 3), dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name,chunk", [("A", 21), ("A", 32), ("C", 48)])
def test_keys_just_inside_and_just_outside_a_chunk(name, chunk, dtype):
    """The needle at a chunk's first position and the probe at its last (the farthest key a row ever sees), the probe at
    the next chunk's first position (the needle has just gone out of sight), and the two on either side of an edge.
    Chunks that end inside a page and at a page's border."""
    c0 = 2 * chunk
    for at, distance, seen in ((c0, chunk - 1, True), (c0, chunk, False), (c0 + chunk - 1, 1, False), (c0 + chunk - 2, 1, True)):
        key, cfg, w, w64, ids, want, moved = needle_case(name, dtype, at, distance, "left", chunk)
        assert (moved >= 0.01) if seen else True, (at, distance, moved)
        run_three_ways(key, cfg, w, w64, ids, want, at + distance, TOL[dtype] if not seen else min(TOL[dtype], moved / 3), dtype,
                       tail=chunk + 3)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_prompts_and_wide_heads(dtype):
    """Heads of 64 and 128 channels, prompts over many pages and chunks, then decoded tokens; alone and two requests
    together, the second cut into portions."""
    cfg, w, w64 = model("C", dtype, seed=9)
    key = ("C9", dtype)
    reqs = {"a": H.random_ids(cfg["vocab"], 330, 1), "b": H.random_ids(cfg["vocab"], 215, 2)}
    eng = engine_for(cfg, w, dtype)
    got = FM.run_trace(eng, H.tail_decode_trace(reqs, tail=12))
    FM.check(key, cfg, w64, reqs, got, dtype)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": reqs["a"][:300], "want": list(range(0, 300, 7))},
                                     {"id": "b", "tokens": reqs["b"][:3], "want": [0, 1, 2]}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": reqs["a"][300:301], "want": [0]},
                                     {"id": "b", "tokens": reqs["b"][3:200], "want": list(range(0, 197, 5))}], "end": []},
             {"step": 2, "entries": [{"id": "a", "tokens": reqs["a"][301:], "want": list(range(29))},
                                     {"id": "b", "tokens": reqs["b"][200:], "want": list(range(15))}], "end": ["a", "b"]}]
    got = FM.run_trace(eng, steps)
    FM.check(key, cfg, w64, reqs, got, dtype)
    eng.cache.check()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_decoding_through_captured_steps(dtype):
    """Three requests decode 150 tokens together, over many page borders and chunk edges; steps of single tokens are
    replayed from captured graphs, and every replay is checked."""
    for name in ("A", "C"):
        cfg, w, w64 = model(name, dtype, seed=6)
        reqs = {f"r{i}": H.random_ids(cfg["vocab"], n, 90 + i) for i, n in enumerate([160, 171, 153])}
        eng = engine_for(cfg, w, dtype, max_requests=3)
        steps = [{"step": 0, "entries": [{"id": r, "tokens": ids[:len(ids) - 150], "want": [0]} for r, ids in reqs.items()],
                  "end": []}]
        for t in range(150):
            steps.append({"step": t + 1, "entries": [{"id": r, "tokens": [ids[len(ids) - 150 + t]], "want": [0]}
                                                     for r, ids in reqs.items()], "end": list(reqs) if t == 149 else []})
        got = FM.run_trace(eng, steps)
        assert eng.graph_replays >= 100
        FM.check((name, dtype, 6), cfg, w64, reqs, got, dtype)


def test_generation_command_line_and_replay_program(tmp_path):
    from tiny_inference_server_amd.engine.generate import generate
    cfg, w, w64 = model("A", seed=8)
    bare = copy.deepcopy(cfg)
    for e in bare["layers"]:                   # as a model folder comes: the two ranks are the weight file's to say
        del e["mixer"]["right"]["decay_rank"], e["mixer"]["right"]["gate_rank"]
    folder = FM.write_folder(str(tmp_path / "m"), bare, w)
    prompts = [H.random_ids(cfg["vocab"], n, 80 + i) for i, n in enumerate((13, 1, 30, 6, 21))]
    want = [pf.greedy_generate(cfg, w64, p, 9) for p in prompts]
    out, s = generate(folder, prompts, max_new_tokens=9, temperature=0.0, dtype="float32", max_batch=3, token_budget=12,
                      pool_tokens=192, return_scheduler=True)
    assert out == want and s.peak_running == 3
    out = generate(folder, prompts[:2], max_new_tokens=5, temperature=0.8, top_k=20, top_p=0.9, rep_penalty=1.1, seed=3)
    assert all(len(o) == 5 and all(0 <= t < cfg["vocab"] for t in o) for o in out)
    proc = subprocess.run([sys.executable, "-m", "tiny_inference_server_amd", "--model", folder, "--prompt-ids",
                           ",".join(map(str, prompts[0])), "--max-new-tokens", "9", "--greedy", "--dtype", "float32"],
                          cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stderr[-3000:]
    line = [l for l in proc.stdout.splitlines() if l.startswith("OUTPUT:")][0]
    assert [int(t) for t in line.split()[1:]] == want[0]
    # the replay program: mixed steps on four state slots and pages for the live requests only
    reqs = {f"r{i}": H.random_ids(cfg["vocab"], n, 70 + i) for i, n in enumerate([40, 64, 30, 70, 12, 50])}
    steps, peak = H.mixed_trace(reqs, max_live=4, seed=8)
    for dtype in ("float32", "bfloat16"):
        out_dir = tmp_path / ("out_" + dtype)
        proc = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "trace_run"), "--model", folder, "--dtype", dtype,
                               "--out", str(out_dir), "--max-tokens", str(peak)],
                              input="\n".join(json.dumps(s) for s in steps) + "\n", capture_output=True, text=True, timeout=300)
        assert proc.returncode == 0, proc.stderr[-3000:]
        assert proc.stdout.split() == [x for s in steps for x in ("done", str(s["step"]))]
        got, fed = {}, {r: 0 for r in reqs}
        for s in steps:
            arr = np.fromfile(out_dir / f"{s['step']}.f32", dtype="<f4").reshape(-1, cfg["vocab"])
            row = 0
            for e in s["entries"]:
                for i in e["want"]:
                    got[(e["id"], fed[e["id"]] + i)] = torch.from_numpy(arr[row].copy())
                    row += 1
                fed[e["id"]] += len(e["tokens"])
        assert len(got) == sum(len(v) for v in reqs.values())
        if dtype == "float32":
            assert FM.worst_error("A8", cfg, w64, reqs, got)[0] <= TOL["float32"]
        else:
            errs = FM.errors("A8", cfg, w64, reqs, got)        # (the router chooses here: most rows are not close calls)
            assert errs[len(errs) // 2][0] <= TOL["bfloat16"] / 2


@pytest.mark.parametrize("Hh,G,D,V,seqs", [
    (2, 1, 64, 16, [48]), (4, 2, 128, 40, [63, 47, 1, 64]), (2, 2, 17, 5, [49, 200]), (3, 1, 200, 33, [65]), (1, 1, 256, 16, [96, 50]),
    (2, 1, 130, 16, [48] * 3 + [2] * 70 + [81])])
def test_the_delta_rules_walk_in_chunks(Hh, G, D, V, seqs):
    """Requests of many rows beside requests of few: whole and ragged chunks, channels that fill no tile, strong and no decays, used state
    lines; against 64 bits, and never further off than a few times what the walk row by row is. A row that is not finite reaches
    no row before it."""
    ops = hip_ops("float32")
    g = torch.Generator().manual_seed(sum(seqs) + D)
    n, C = sum(seqs), 2 * G * D + Hh * V
    firsts = [sum(seqs[:i]) for i in range(len(seqs))]
    b = fake_batch([(f, 0, r) for f, r in zip(firsts, seqs)], list(range(len(seqs)))[::-1], None, 8, "cuda")
    k, q = (torch.nn.functional.normalize(torch.randn(n, G, D, generator=g), dim=-1) for _ in range(2))
    v, beta = torch.randn(n, Hh * V, generator=g), torch.rand(n, Hh, generator=g)
    decay = torch.exp(-torch.rand(n, Hh * D, generator=g) * torch.rand(1, Hh * D, generator=g) * 3.0)
    decay[n // 2, :D // 2] = 0.0
    decay[:, D // 2:D] = 1.0
    blocks = -(-V // 16)
    line = torch.zeros(len(seqs), Hh, blocks, D, 16)
    line.permute(0, 1, 3, 2, 4).reshape(len(seqs), Hh, D, blocks * 16)[..., :V]
    start = torch.randn(len(seqs), Hh, D, V, generator=g)
    for c in range(V):
        line[:, :, c // 16, :, c % 16] = start[..., c]

    def engine(v):
        state = line.reshape(len(seqs), -1).clone().cuda()
        u = torch.cat([(q * D ** -0.5).reshape(n, -1), k.reshape(n, -1), v, beta], 1).cuda()
        out = ops.delta_scan(u, 0, G * D, 2 * G * D, C, decay.cuda(), state, b, Hh, G, D, V)
        return out.cpu(), state.cpu().view(len(seqs), Hh, blocks, D, 16)

    def plain(dt):
        out, end = torch.empty(n, Hh, V, dtype=dt), start.to(dt).flip(0).clone()
        kk, qq = (t.to(dt).repeat_interleave(Hh // G, 1) for t in (k, q * D ** -0.5))
        for i, (f, r) in enumerate(zip(firsts, seqs)):
            S = end[i]
            for t in range(f, f + r):
                S = S * decay[t].to(dt).view(Hh, D, 1)
                w = beta[t].to(dt)[:, None, None] * (v[t].to(dt).view(Hh, 1, V) - kk[t][:, None] @ S)
                S = S + kk[t][:, :, None] * w
                out[t] = (qq[t][:, None] @ S)[:, 0]
            end[i] = S
        return out.reshape(n, -1), end.flip(0)

    out, state = engine(v)
    want, end = plain(torch.float64)
    near, near_end = plain(torch.float32)
    kept = torch.stack([state[:, :, c // 16, :, c % 16] for c in range(V)], -1)
    for got, exact, row in ((out, want, near), (kept, end, near_end)):
        off = lambda t: float((t.double() - exact).norm() / exact.norm())
        assert off(got) <= 3 * off(row) + 1e-7, (off(got), off(row))
    for c in range(V, blocks * 16):
        assert (state[:, :, c // 16, :, c % 16] == 0).all()
    longest = max(range(len(seqs)), key=lambda i: seqs[i])
    at = firsts[longest] + 37
    bad = v.clone()
    bad[at] = float("inf")
    broken, _ = engine(bad)
    before = torch.ones(n, dtype=torch.bool)
    before[at:firsts[longest] + seqs[longest]] = False
    torch.testing.assert_close(broken[before], out[before], rtol=1e-4, atol=1e-5)
    assert not torch.isfinite(broken[at]).any()


@pytest.mark.parametrize("K", [1, 2, 4, 7])
@pytest.mark.parametrize("seq_rows,slots", [([(0, 40, 1)], [2]), ([(i, 3 * i, 1) for i in range(70)], list(range(70))[::-1]), ([(0, 5, 1), (1, 0, 9), (10, 7, 2)], [1, 0, 2])])
def test_single_rows_move_their_lines_on_with_the_step_before_the_walk(seq_rows, slots, K):
    """The bits of the two kernels, in what is prepared and in every line; requests of more rows go to both as before."""
    ops, g = hip_ops("float32"), torch.Generator().manual_seed(K + len(slots))
    Hh, G, D, V, off = 4, 2, 70, 24, 3
    C, n = 2 * G * D + Hh * V, sum(r[2] for r in seq_rows)
    taps, proj = torch.randn(C, K, generator=g).cuda(), torch.randn(n, off + C + Hh, generator=g).cuda()
    b, at = fake_batch(seq_rows, slots, None, 8, "cuda"), Hh * 2 * D * 16
    lines = [torch.randn(max(slots) + 1, at + (K - 1) * C + 4, generator=g).cuda()]
    lines.append(lines[0].clone())
    one = ops.delta_prepare_and_keep(proj, off, off + C, taps, lines[0], at, b, Hh, G, D, V)
    two = ops.delta_prepare(proj, off, off + C, taps, lines[1], at, b, Hh, G, D, V)
    ops.conv_state_update(proj, off, C, K, lines[1], at, b)
    assert torch.equal(one, two) and torch.equal(*lines)


@pytest.mark.parametrize("n,ranks,widths", [(1, (64, 64), (1024, 2048)), (5, (16, 9), (512, 100)), (257, (64, 64), (1000, 2048)), (300, (64, 40), (1024, 2048)),
                                            (33, (130, 16), (96, 33)), (300, (33, 64), (1024, 1024))])
def test_two_low_rank_products_in_one_launch(n, ranks, widths):
    """Each the bits of its own launch: of one form, and of two (another chunk of the rank, another number of rows a thread, lines read 16 bytes at a time or not)."""
    ops, g = hip_ops("float32"), torch.Generator().manual_seed(n)
    low = torch.randn(n, sum(ranks) + 4, generator=g).cuda()
    w = [torch.randn(c, r, generator=g).cuda() for c, r in zip(widths, ranks)]
    bias, rate = torch.randn(widths[0], generator=g).cuda(), torch.rand(widths[0], generator=g).cuda()
    first = dict(low=low[:, :ranks[0]], w2=w[0], bias=bias, kind="exp_softplus", rate=rate, group=1)
    second = dict(low=low[:, ranks[0]:ranks[0] + ranks[1]], w2=w[1], bias=None, kind="none")
    for a, b in ((first, second), (second, first)):
        got = ops.lowrank_act_pair(a, b)
        assert torch.equal(got[0], ops.lowrank_act(**a)) and torch.equal(got[1], ops.lowrank_act(**b))
    from tiny_inference_server_amd.ops.hip_ops import KernelError
    with pytest.raises(KernelError):
        ops.lowrank_act_pair(first, dict(second, low=second["low"][:n - 1]))


@pytest.mark.parametrize("D", [64, 130])
def test_a_walk_in_chunks_gives_a_prefix_its_own_bits(D):
    """Whatever number of chunks follows, and however many of them the last turn of the loop takes: the rows before get the same bits, whole chunks and
    begun ones."""
    Hh, G, V, n = 2, 1, 24, 163
    ops = hip_ops("float32")
    g = torch.Generator().manual_seed(D)
    C = 2 * G * D + Hh * V
    k, q = (torch.nn.functional.normalize(torch.randn(n, G, D, generator=g), dim=-1) for _ in range(2))
    u = torch.cat([(q * D ** -0.5).reshape(n, -1), k.reshape(n, -1), torch.randn(n, Hh * V, generator=g), torch.rand(n, Hh, generator=g)], 1).cuda()
    decay = torch.exp(-torch.rand(n, Hh * D, generator=g)).cuda()
    start = torch.randn(1, Hh * 2 * D * 16, generator=g).cuda()

    def rows(m):
        return ops.delta_scan(u[:m], 0, G * D, 2 * G * D, C, decay[:m], start.clone(), fake_batch([(0, 0, m)], [0], None, 8, "cuda"), Hh, G, D, V)
    whole = rows(n)
    for m in (48, 49, 63, 64, 65, 80, 95, 96, 112, 128, 129, 144, 160):
        assert torch.equal(rows(m), whole[:m]), m


# Rows walked in chunks against the walk row by row, both against 64 bits: the chunks add the same products up in sums of no more terms and
# in the rows' order, so neither results nor states lie further off. Either error is the norm of some 100,000 independent roundings of
# which every one weighs the same, so the two would differ by 1 % if their roundings were as many; 8 % leaves room for T, which
# the walk row by row does not have (chunks whose products took rows out of their order: 12 to 35 %).
@pytest.mark.parametrize("H,G,D,V", [(8, 4, 128, 256), (4, 2, 64, 64), (2, 2, 200, 48)])
@pytest.mark.parametrize("least", [0.5, 0.9, 0.995])
def test_the_delta_rule_in_chunks_is_no_further_off_than_row_by_row(monkeypatch, H, G, D, V, least):
    from tiny_inference_server_amd.ops import hip_ops as module
    ops, n, blocks = hip_ops("float32"), 300, V // 16
    g = torch.Generator().manual_seed(D)
    qk = torch.nn.functional.normalize(torch.randn(n, 2 * G, D, generator=g), dim=-1)
    qk[:, :G] *= D ** -0.5
    u = torch.cat((qk.reshape(n, -1), torch.nn.functional.silu(torch.randn(n, H * V, generator=g)), torch.rand(n, H, generator=g)), 1).cuda()
    decay = (least + (1 - least) * torch.rand(n, H * D, generator=g)).cuda()
    line = (0.3 * torch.randn(1, H * blocks * D * 16, generator=g)).cuda()
    as_state = lambda t: t.view(H, blocks, D, 16).permute(0, 2, 1, 3).reshape(H, D, V)
    S, C, want = as_state(line).double(), 2 * G * D + H * V, []
    wide, slow = u.double(), decay.double()
    for r in range(n):
        q, k = (wide[r, i * G * D:(i + 1) * G * D].view(G, D).repeat_interleave(H // G, 0) for i in (0, 1))
        S = S * slow[r].view(H, D, 1)
        w = wide[r, C:, None] * (wide[r, 2 * G * D:C].view(H, V) - (S * k[:, :, None]).sum(1))
        S = S + k[:, :, None] * w[:, None]
        want.append((S * q[:, :, None]).sum(1).reshape(-1))
    want, off = torch.stack(want), []
    for most in (0, module._DELTA_WORK_FLOATS):      # without work space: row by row
        monkeypatch.setattr(module, "_DELTA_WORK_FLOATS", most)
        st = line.clone()
        out = ops.delta_scan(u, 0, G * D, 2 * G * D, C, decay, st, fake_batch([(0, 0, n)], [0], None, 1, "cuda"), H, G, D, V)
        off.append([((a.double() - b).norm() / b.norm()).item() for a, b in ((out, want), (as_state(st), S))])
    assert all(chunks <= 1.08 * rows for rows, chunks in zip(*off)), off


@pytest.mark.parametrize("lens,chunks", [([1] * 64, False), ([47, 47], False), ([48], True), ([1] * 20 + [48], True)])
def test_the_delta_rule_asks_for_chunks_only_where_a_request_is_long(lens, chunks):
    """Single tokens of 64 requests are many rows and no long request: the call takes no memory beyond its result (the chunks' operands
    would be megabytes, and two kernels would be launched for them); one request of 48 rows does."""
    ops = hip_ops("float32")
    H, D, V, n = 4, 64, 32, sum(lens)
    firsts = [sum(lens[:i]) for i in range(len(lens))]
    b = fake_batch([(f, 0, r) for f, r in zip(firsts, lens)], list(range(len(lens))), None, 8, "cuda")
    C = 2 * H * D + H * V
    u, decay = torch.randn(n, C + H, device="cuda"), torch.rand(n, H * D, device="cuda")
    state = torch.zeros(len(lens), H * V * D, device="cuda")
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = ops.delta_scan(u, 0, H * D, 2 * H * D, C, decay, state, b, H, H, D, V)
    more = torch.cuda.max_memory_allocated() - before - out.numel() * 4
    assert (more > 4096) == chunks, more
