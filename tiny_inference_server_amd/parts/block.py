"""Arrangements: how a block wires its norms, its mixer and its feed-forward."""
from __future__ import annotations

from .base import ARRANGEMENTS, Arrangement, states


@ARRANGEMENTS.register("prenorm_residual")
class PreNormResidual(Arrangement):
    """x = x + mixer(norm_a(x)); x = x + feed_forward(norm_f(x))   (reference main_models_new.py:146-152)."""
    part_names = ("mixer_norm", "mixer", "feed_forward_norm", "feed_forward")

    def __init__(self, layer_spec, tensors, ops):
        super().__init__(layer_spec, tensors, ops)
        self.mixer_norm, self.mixer = self.parts["mixer_norm"], self.parts["mixer"]
        self.ffn_norm, self.ffn = self.parts["feed_forward_norm"], self.parts["feed_forward"]
        # a block of parts that say what they are made of may be one kernel, where the operations object has it and takes the step
        self.one_kernel = ops.small_block if (getattr(ops, "small", None) is not None and states(self.mixer, "whole_block") and states(self.ffn, "whole_block")
                                              and hasattr(self.mixer_norm, "as_rms") and hasattr(self.ffn_norm, "as_rms")) else None

    def forward(self, x, ctx):
        # the stream `x` is replaced by each sub-layer's result, so the residual passed down is spent and a part may
        # write its result over it; whether the block's own input is spent too, the caller says in ctx
        mctx = ctx.of("mixer")
        mixer = self.mixer.whole_block(mctx) if self.one_kernel is not None else None
        if mixer is not None:
            y = self.one_kernel(x, mctx.batch, mctx.group, mctx.plane, (self.mixer_norm.as_rms(), self.ffn_norm.as_rms()), mixer, self.ffn.whole_block())
            if y is not None:
                return y
        if getattr(self.mixer, "fuses_norm", False):
            x = self.mixer.forward(x, mctx, residual=x, norm=self.mixer_norm)
        else:
            x = self.mixer.forward(self.mixer_norm(x), mctx, residual=x)
        if getattr(self.ffn, "fuses_norm", False):
            return self.ffn.forward(x, residual=x, norm=self.ffn_norm, residual_is_spent=True)
        return self.ffn.forward(self.ffn_norm(x), residual=x)
