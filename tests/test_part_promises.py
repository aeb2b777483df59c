"""What a part's class says of itself holds for that class and for none derived from it; and which of a block's two mixers goes beside the other. On the host,
with a stand-in for the operations that only a GPU has."""
from __future__ import annotations

import dataclasses
from types import SimpleNamespace

import pytest
import torch

from tiny_inference_server_amd.architectures.gqa_mtp import build_spec
from tiny_inference_server_amd.config import ARCHITECTURES, Architecture, GqaMtpConfig
from tiny_inference_server_amd.engine import Engine
from tiny_inference_server_amd.ops.hip_ops import HipOps
from tiny_inference_server_amd.parts import FEED_FORWARDS, MIXERS
from tiny_inference_server_amd.parts.attention import GqaAttention
from tiny_inference_server_amd.parts.base import side_by_side
from tiny_inference_server_amd.parts.feed_forward import SwiGlu
from tiny_inference_server_amd.parts.recurrent import GatedDeltaRule, GatedLinearAttention, LightningAttention, MatrixMemory
from tiny_inference_server_amd.weights import random_tensors
from torch_ops import TorchOps

CFG = GqaMtpConfig(d_model=64, vocab_size=97, max_context=128, rope_base=1e4, n_heads=8, n_layers=2, ffn_hidden=176, group_size=4, mtp_heads=0,
                   architecture="PromisesToy")


class _Blocks(TorchOps):
    """Operations that take a whole block, and count it, by way of the separate ones."""
    small = object()

    def __init__(self):
        super().__init__()
        self.blocks = 0

    def small_block(self, x, batch, group, plane, norms, attention, feed_forward):
        if batch.max_seq_rows > 1:
            return None
        self.blocks += 1
        w_qkv, w_o, table, interleaved, H, G, HD, window, scale = attention
        q = self.qkv_rope(x, w_qkv, norms[0], batch.positions, batch.write_slots[group], table, plane, H, G, HD, plane.shape[3], interleaved)
        mid = self.linear(self.paged_attention(q, plane, batch, group, H, G, HD, window, scale), w_o, residual=x)
        return self.linear(self.linear_swiglu(mid, feed_forward[0], rms=norms[1]), feed_forward[1], residual=mid)


class _Doubled(GqaAttention):
    """Attention whose output projection is applied twice as large."""
    calls = 0

    def forward(self, x, ctx, residual=None, norm=None):
        type(self).calls += 1
        y = super().forward(x, ctx, None, norm)
        return residual + 2.0 * y


class _Halved(SwiGlu):
    calls = 0

    def forward(self, x, residual=None, norm=None, residual_is_spent=False):
        type(self).calls += 1
        return residual + 0.5 * super().forward(x, None, norm)


@pytest.mark.parametrize("role,kind", [("mixer", _Doubled), ("feed_forward", _Halved), (None, None)])
def test_a_derived_part_runs_in_every_step(role, kind):
    """A part derived from one that a whole block's kernel knows, with a computation of its own: it is called in steps of single rows as in the prompt, so
    a sequence has the same logits fed at once and token by token. The parts themselves go to that kernel."""
    MIXERS.register("_doubled", _Doubled, replace=True)
    FEED_FORWARDS.register("_halved", _Halved, replace=True)

    def spec(cfg):
        base = build_spec(cfg)
        if role is None:
            return base
        layers = tuple(b.with_part(role, dataclasses.replace(b.part(role), kind={"mixer": "_doubled", "feed_forward": "_halved"}[role])) for b in base.layers)
        return dataclasses.replace(base, layers=layers)
    ARCHITECTURES.register("PromisesToy", Architecture("PromisesToy", GqaMtpConfig, spec), replace=True)
    try:
        ops = _Blocks()
        eng = Engine(config=CFG, tensors=random_tensors(CFG, 5, std=0.1, dtype="float32"), dtype="float32", page_size=16, max_tokens=128, max_requests=2, ops=ops)
        ids = torch.randint(0, 97, (9,), generator=torch.Generator().manual_seed(1)).tolist()
        whole = eng.step([("a", ids, range(9))]).logits.clone()
        if kind is not None:
            kind.calls = 0
        single = torch.cat([eng.step([("b", [t], [0])]).logits.clone() for t in ids])
        torch.testing.assert_close(single, whole, rtol=1e-4, atol=1e-4)
        if kind is None:
            assert ops.blocks == 9 * CFG.n_layers
        else:
            assert ops.blocks == 0 and kind.calls == 9 * CFG.n_layers
    finally:
        ARCHITECTURES.unregister("PromisesToy")
        MIXERS.unregister("_doubled")
        FEED_FORWARDS.unregister("_halved")


class _Streams:
    def __init__(self, pays=True):
        self.pays, self.log = pays, []

    def beside_pays(self, batch, width):
        return self.pays and width == 7

    def beside(self, first, second):
        self.log.append(("beside", second()))
        self.log.append(("here", first()))
        return self.log[-1][1], self.log[-2][1]


class _Own:
    own_memory = True


class _Shared:
    pass


class _FromOwn(_Own):
    """(what it adds may use the shared work space)"""


@pytest.mark.parametrize("left,right,beside", [(_Shared, _Own, "right"), (_Own, _Shared, "left"), (_Own, _Own, "right"), (_Shared, _Shared, None),
                                               (_Shared, _FromOwn, None), (_FromOwn, _Shared, None)])
@pytest.mark.parametrize("pays", [True, False])
def test_which_mixer_goes_beside_the_other(left, right, beside, pays):
    """The one that owns its memory, whichever side it is on; results come in the order of the calls."""
    ops = _Streams(pays)
    assert side_by_side(ops, None, 7, [(left(), lambda: "left"), (right(), lambda: "right")]) == ["left", "right"]
    if pays and beside:
        assert ops.log == [("beside", beside), ("here", "left" if beside == "right" else "right")]
    else:
        assert ops.log == []
    assert side_by_side(ops, None, 7, [(_Own(), lambda: 1)]) == [1] and side_by_side(object(), None, 7, [(_Own(), lambda: 1), (_Own(), lambda: 2)]) == [1, 2]


@pytest.mark.parametrize("width,captured,launched", [(512, 1024, 6144), (1024, 256, 3072), (1408, 136, 2235), (2048, 64, 1536), (4096, 64, 1536)])
def test_rows_from_which_mixers_run_side_by_side(width, captured, launched, monkeypatch):
    """More of them the narrower the model is, as it has less to do in the same launches."""
    ops = SimpleNamespace(dtype=torch.bfloat16)
    for capturing, first in ((True, captured), (False, launched)):
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
        assert [HipOps.beside_pays(ops, SimpleNamespace(max_seq_rows=n), width) for n in (1, first - 1, first, first + 5000)] == [False, False, True, True]
    assert not HipOps.beside_pays(SimpleNamespace(dtype=torch.float32), SimpleNamespace(max_seq_rows=9999), width)


def test_mixers_that_own_their_memory():
    assert all(c.__dict__.get("own_memory") is True for c in (GatedDeltaRule, GatedLinearAttention, LightningAttention, MatrixMemory))
