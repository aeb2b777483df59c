"""Attention mixers."""
from __future__ import annotations

import torch

from .base import MIXERS, build_part, layer_product, to_compute
from .spec import PagedKvNeed, StateNeed


@MIXERS.register("gqa_attention")
class GqaAttention:
    """Grouped-query attention over a paged cache.

    q = x.Wq, [k|v] = x.Wkv, rotary on q and k, keys and values written into the call's cache plane before
    any row attends, then every row at position p attends the keys [0, p] (or the last `window`) of its
    own request, query head h using key/value head h // group_size; out = attn.Wo (+ residual)
    (reference main_models_new.py:96-136; paged_attention_kernels.py:49).

    params: d_model, n_heads, n_kv_heads, head_dim, window (0: all keys), position (a PartSpec).
    tensors: q (d_model, n_heads*head_dim), kv (d_model, 2*n_kv_heads*head_dim) with the key columns first,
    o (n_heads*head_dim, d_model); all stored [in, out] as the reference applies them (x @ W).
    """
    graph_safe = True

    @classmethod
    def tensor_shapes(cls, params):
        d, nh, nkv, hd = params["d_model"], params["n_heads"], params["n_kv_heads"], params["head_dim"]
        return {"q": (d, nh * hd), "kv": (d, 2 * nkv * hd), "o": (nh * hd, d)}

    @classmethod
    def cache_need(cls, params):
        return PagedKvNeed(params["n_kv_heads"], params["head_dim"], int(params.get("window", 0)))

    def __init__(self, spec, tensors, ops):
        p = spec.params
        self.ops = ops
        self.n_heads, self.n_kv_heads, self.head_dim = int(p["n_heads"]), int(p["n_kv_heads"]), int(p["head_dim"])
        if self.n_heads % self.n_kv_heads:
            raise ValueError(f"{self.n_heads} query heads are not a multiple of {self.n_kv_heads} key/value heads")
        self.window = int(p.get("window", 0))
        self.scale = float(p.get("scale", self.head_dim ** -0.5))
        pos = p["position"]
        self.position = build_part(pos, tensors, ops)
        # a position encoding may work on the scores instead of (or beside) rotating queries and keys
        slopes = getattr(self.position, "score_slopes", None)
        self.slopes = slopes(self.n_heads) if slopes is not None else None
        # one projection for q, k and v: rows of the [out, in] matrix are q heads, then k heads, then v heads.
        # Inside every q and k head the rows are put in pair order (the two members of a rotary pair side by side),
        # so that the kernel that makes them can rotate them while they are still in its registers.
        w = torch.cat((tensors.of(spec, "q"), tensors.of(spec, "kv")), dim=1).t()
        _, interleaved = self.position.rotary()
        hd, half = self.head_dim, self.head_dim // 2
        if not interleaved:
            order = torch.stack((torch.arange(half), torch.arange(half) + half), dim=1).reshape(-1)
            rows = torch.arange(w.shape[0]).view(-1, hd)
            n_qk = self.n_heads + self.n_kv_heads
            rows[:n_qk] = rows[:n_qk][:, order]
            w = w[rows.reshape(-1)]
        self.w_qkv = to_compute(ops, w)
        self.w_o = to_compute(ops, tensors.of(spec, "o").t())
        self.q_width = self.n_heads * self.head_dim

    fuses_norm = True

    def whole_block(self, ctx):
        """What an operations object's kernel for whole small blocks takes of this mixer (HipOps.small_block); None where it is more than that."""
        if self.slopes is not None or not ctx.writes_cache:
            return None
        return (self.w_qkv, self.w_o, *self.position.rotary(), self.n_heads, self.n_kv_heads, self.head_dim, self.window, self.scale)

    # work lists for the attention kernels are made on the host, once per step and attention shape
    def plan_key(self):
        if not hasattr(self.ops, "plan_attention"):
            return None
        return ("attention", self.n_heads, self.n_kv_heads, self.head_dim, self.window)

    def plan_mode(self, seq_rows):
        mode = getattr(self.ops, "plan_attention_mode", None)
        return mode(seq_rows, self.window) if mode is not None else None

    def plan_rows(self, seq_rows, add, mode=None):
        return self.ops.plan_attention(self.n_heads, self.n_kv_heads, self.head_dim, seq_rows, add, mode, self.window)

    def forward(self, x, ctx, residual=None, norm=None):
        ops, b = self.ops, ctx.batch
        rms = None
        if norm is not None:
            if hasattr(norm, "as_rms"):
                rms = norm.as_rms()
            else:
                x = norm(x)
        table, interleaved = self.position.rotary()
        page_size = ctx.plane.shape[3]
        q = ops.qkv_rope(x, self.w_qkv, rms, b.positions, b.write_slots[ctx.group], table, ctx.plane, self.n_heads,
                         self.n_kv_heads, self.head_dim, page_size, interleaved, ctx.writes_cache)
        extra = {"slopes": self.slopes} if self.slopes is not None else {}
        attn = ops.paged_attention(q, ctx.plane, b, ctx.group, self.n_heads, self.n_kv_heads,
                                   self.head_dim, self.window, self.scale, **extra)
        return layer_product(ops)(attn, self.w_o, residual=residual, reuse_residual=ctx.residual_is_spent)


@MIXERS.register("windowed_qknorm_attention")
class WindowedQkNormAttention:
    """Grouped-query softmax attention over the last `window` positions (0: all), with keys and values of different
    sizes. q = x.Wq^T, k = x.Wk^T, v = x.Wv^T; queries and keys are RMS-normed per head (a gain of key_dim entries
    each, shared by the heads), then the first rot_dims channels of each head are rotated in interleaved pairs
    (2i, 2i+1) by position * base^(-2i/rot_dims); values are divided by their root mean square and cached so;
    score = q.k * scale * temp[head]; out = softmax-weighted values of all heads . Wo^T. Norms, angles, scores and
    the softmax are 32-bit.

    params: width, n_heads, n_kv_heads, key_dim, value_dim, window, rot_dims, rot_base, scale, eps. tensors, stored
    [out, in]: q (heads*key_dim, width), k (kv_heads*key_dim, width), v (kv_heads*value_dim, width), q_norm, k_norm
    (key_dim,), temp (heads,), o (width, heads*value_dim).
    """
    graph_safe = True

    @classmethod
    def tensor_shapes(cls, params):
        w, H, G, kd, vd = (params[k] for k in ("width", "n_heads", "n_kv_heads", "key_dim", "value_dim"))
        return {"q": (H * kd, w), "k": (G * kd, w), "v": (G * vd, w), "q_norm": (kd,), "k_norm": (kd,), "temp": (H,),
                "o": (w, H * vd)}

    @classmethod
    def cache_need(cls, params):
        return PagedKvNeed(params["n_kv_heads"], params["key_dim"], int(params.get("window", 0)),
                           value_dim=params["value_dim"])

    def __init__(self, spec, tensors, ops):
        from .base import to_gain
        p = spec.params
        self.ops = ops
        self.H, self.G, self.kd, self.vd = int(p["n_heads"]), int(p["n_kv_heads"]), int(p["key_dim"]), int(p["value_dim"])
        if self.H % self.G:
            raise ValueError(f"{self.H} query heads are not a multiple of {self.G} key/value heads")
        self.window, self.scale, self.eps = int(p.get("window", 0)), float(p["scale"]), float(p["eps"])
        self.rot_dims = int(p.get("rot_dims", 0))
        if self.rot_dims % 2 or self.rot_dims > self.kd:
            raise ValueError(f"{self.rot_dims} rotated channels of a head of {self.kd}: an even number, at most the head")
        i = torch.arange(self.rot_dims // 2, dtype=torch.float64)
        self.freqs = (float(p.get("rot_base", 10000.0)) ** (-2.0 * i / max(1, self.rot_dims))).to(torch.float32).to(ops.device)
        q, k, v = tensors.of(spec, "q"), tensors.of(spec, "k"), tensors.of(spec, "v")
        self.input_rows = torch.cat((q, k, v), dim=0)
        self.k_at, self.v_at = q.shape[0], q.shape[0] + k.shape[0]
        self._w_in = None
        self.q_gain, self.k_gain = to_gain(ops, tensors.of(spec, "q_norm")), to_gain(ops, tensors.of(spec, "k_norm"))
        self.temp = to_gain(ops, tensors.of(spec, "temp"))
        self.w_o = to_compute(ops, tensors.of(spec, "o"))
        self.same = self.kd == self.vd        # then the pages have the layout every attention kernel reads

    # the matrix-core kernels' work lists, where keys and values are of one size (see GqaAttention)
    def plan_key(self):
        if not self.same or not hasattr(self.ops, "plan_attention"):
            return None
        return ("attention", self.H, self.G, self.kd, self.window)

    def plan_mode(self, seq_rows):
        mode = getattr(self.ops, "plan_attention_mode", None)
        return mode(seq_rows, self.window) if mode is not None and self.same else None

    def plan_rows(self, seq_rows, add, mode=None):
        return self.ops.plan_attention(self.H, self.G, self.kd, seq_rows, add, mode, self.window)

    def core(self, proj, ctx):
        ops, b = self.ops, ctx.batch
        q = ops.attention_prepare(proj, 0, self.k_at, self.v_at, b.positions, b.write_slots[ctx.group], ctx.plane, self.H,
                                  self.G, self.kd, self.vd, ctx.page_size, self.q_gain, self.k_gain, self.temp,
                                  self.freqs, self.rot_dims, self.eps, ctx.writes_cache)
        if self.same:
            return ops.paged_attention(q, ctx.plane, b, ctx.group, self.H, self.G, self.kd, self.window, self.scale)
        return ops.paged_attention_kv(q, ctx.plane, b, ctx.group, self.H, self.G, self.kd, self.vd, ctx.page_size,
                                      self.window, self.scale)

    def forward_projected(self, proj, ctx):
        return self.ops.linear(self.core(proj, ctx), self.w_o, out_dtype=torch.float32)

    def forward(self, x, ctx, residual=None):
        if self._w_in is None:
            self._w_in = to_compute(self.ops, self.input_rows)
        proj = self.ops.linear(x, self._w_in, out_dtype=torch.float32)
        return self.ops.linear(self.core(proj, ctx), self.w_o, residual=residual)


def banded_frequencies(dims: int, base: float, bands=None):
    """base^(-2i/dims) for the pairs i < dims/2 in 64-bit. bands = (factor, low, high, original) slows the long waves:
    with wavelength l = 2 pi / f, a pair with l < original / high keeps f, one with l > original / low turns at
    f / factor, and between the two f is blended with f / factor by s = (original / l - low) / (high - low):
    (1 - s) f / factor + s f."""
    import math
    i = torch.arange(dims // 2, dtype=torch.float64)
    f = float(base) ** (-2.0 * i / max(1, dims))
    if bands is None:
        return f
    factor, low, high, original = (float(b) for b in bands)
    wave = 2.0 * math.pi / f
    if high == low:
        s = (wave < original / high).to(torch.float64)
    else:
        s = torch.clamp((original / wave - low) / (high - low), 0.0, 1.0)
    blended = (1.0 - s) * f / factor + s * f
    return torch.where(wave < original / high, f, torch.where(wave > original / low, f / factor, blended))


def _rotary_frequencies(ops, dims: int, base: float, bands=None):
    """The rotation's frequencies on the device in 32-bit (computed in 64-bit)."""
    return banded_frequencies(dims, base, bands).to(torch.float32).to(ops.device)


def slowed_frequencies(dims: int, base: float, factor: float, original: float, fast: float, slow: float):
    """(frequencies in 64-bit, factor on cosine and sine) of a rotation whose long waves are slowed by `factor`.

    A pair that turns n times within `original` positions sits at i(n) = dims ln(original / (2 pi n)) / (2 ln base). Up to
    pair floor(i(fast)) the frequencies base^(-2i/dims) are kept, from pair ceil(i(slow)) on they are divided by `factor`,
    and linearly blended between the two (both clamped to 0 .. dims - 1; where they coincide, a step)."""
    import math
    f = banded_frequencies(dims, base)
    at = [dims * math.log(original / (2.0 * math.pi * n)) / (2.0 * math.log(base)) for n in (fast, slow)]
    lo, hi = max(math.floor(at[0]), 0), min(math.ceil(at[1]), dims - 1)
    ramp = torch.clamp((torch.arange(dims // 2, dtype=torch.float64) - lo) / max(hi - lo, 0.001), 0.0, 1.0)
    return f / factor * ramp + f * (1.0 - ramp), 0.1 * math.log(factor) + 1.0


def _rotation(ops, dims: int, base: float, slowed=None):
    """(frequencies on the device in 32-bit, factor on cosine and sine); slowed: (factor, original, fast, slow) or None."""
    if slowed is None or not dims:
        return _rotary_frequencies(ops, dims, base), 1.0
    f, factor = slowed_frequencies(dims, base, *(float(v) for v in slowed))
    return f.to(torch.float32).to(ops.device), factor


def stacked_rows(mats):
    """(the matrices one below the other, each starting at a multiple of 8 rows; their first rows): the columns of a
    32-bit product with them then start 32 bytes apart."""
    blocks, starts, at = [], [], 0
    for m in mats:
        pad = -m.shape[0] % 8
        starts.append(at)
        blocks.append(m)
        if pad:
            blocks.append(torch.zeros(pad, m.shape[1], dtype=m.dtype, device=m.device))
        at += m.shape[0] + pad
    return torch.cat(blocks, dim=0), starts


@MIXERS.register("sink_gated_attention")
class SinkGatedAttention:
    """Grouped-query attention over all earlier positions with biased projections, no rotation, a query factor that
    grows with the position, a sink in the softmax and a gate per head.

    q = x.Wq^T + bq, k = x.Wk^T + bk, v = x.Wv^T + bv; the query at position p is multiplied by
    1 + temp_coef * ln(floor((p + 1) / temp_every) + 1); score = q.k * scale; the weights of a row are
    exp(s_j) / (1 + sum_j exp(s_j)) (a sink of score 0 without a value); head h's result is multiplied by
    sigmoid(x.Wg^T)[h]; out = heads . Wo^T. Factors, scores, weights and gates are 32-bit. Keys and values may differ in
    size.

    params: width, n_heads, n_kv_heads, key_dim, value_dim, scale, temp_coef, temp_every (temp_coef 0: no factor),
    sink (default true), head_gate (default true). tensors, stored [out, in]: q (heads*key_dim, width), k
    (kv_heads*key_dim, width), v (kv_heads*value_dim, width), q_bias, k_bias, v_bias, g (heads, width; with head_gate),
    o (width, heads*value_dim).
    """
    graph_safe = True

    @classmethod
    def tensor_shapes(cls, params):
        w, H, G, kd, vd = (params[k] for k in ("width", "n_heads", "n_kv_heads", "key_dim", "value_dim"))
        shapes = {"q": (H * kd, w), "k": (G * kd, w), "v": (G * vd, w), "q_bias": (H * kd,), "k_bias": (G * kd,),
                  "v_bias": (G * vd,), "o": (w, H * vd)}
        if params.get("head_gate", True):
            shapes["g"] = (H, w)
        return shapes

    @classmethod
    def cache_need(cls, params):
        return PagedKvNeed(params["n_kv_heads"], params["key_dim"], 0, value_dim=params["value_dim"])

    def __init__(self, spec, tensors, ops):
        from .base import to_gain
        p = spec.params
        self.ops = ops
        self.H, self.G, self.kd, self.vd = int(p["n_heads"]), int(p["n_kv_heads"]), int(p["key_dim"]), int(p["value_dim"])
        if self.H % self.G:
            raise ValueError(f"{self.H} query heads are not a multiple of {self.G} key/value heads")
        self.scale = float(p["scale"])
        self.temp_coef, self.temp_every = float(p.get("temp_coef", 0.0)), int(p.get("temp_every", 1))
        self.sink, self.head_gate = bool(p.get("sink", True)), bool(p.get("head_gate", True))
        mats = [tensors.of(spec, k) for k in ("q", "k", "v")] + ([tensors.of(spec, "g")] if self.head_gate else [])
        self.k_at = mats[0].shape[0]
        self.v_at = self.k_at + mats[1].shape[0]
        self.g_at = self.v_at + mats[2].shape[0]
        self.w_in = to_compute(ops, torch.cat(mats, dim=0))
        self.q_bias, self.k_bias, self.v_bias = (to_gain(ops, tensors.of(spec, k)) for k in ("q_bias", "k_bias", "v_bias"))
        self.w_o = to_compute(ops, tensors.of(spec, "o"))
        self.same = self.kd == self.vd        # then the pages have the layout every attention kernel reads

    # the matrix-core kernels' work lists, where keys and values are of one size (see GqaAttention)
    def plan_key(self):
        if not self.same or not hasattr(self.ops, "plan_attention"):
            return None
        return ("attention", self.H, self.G, self.kd, 0)

    def plan_mode(self, seq_rows):
        mode = getattr(self.ops, "plan_attention_mode", None)
        return mode(seq_rows, 0) if mode is not None and self.same else None

    def plan_rows(self, seq_rows, add, mode=None):
        return self.ops.plan_attention(self.H, self.G, self.kd, seq_rows, add, mode, 0)

    def core(self, x, ctx):
        ops, b = self.ops, ctx.batch
        proj = ops.linear(x, self.w_in, out_dtype=torch.float32)
        q = ops.attention_prepare(proj, 0, self.k_at, self.v_at, b.positions, b.write_slots[ctx.group], ctx.plane, self.H,
                                  self.G, self.kd, self.vd, ctx.page_size, write_cache=ctx.writes_cache, value_norm=False,
                                  q_bias=self.q_bias, k_bias=self.k_bias, v_bias=self.v_bias, temp_coef=self.temp_coef,
                                  temp_every=self.temp_every)
        gate = proj[:, self.g_at:self.g_at + self.H] if self.head_gate else None
        if self.same:
            return ops.paged_attention(q, ctx.plane, b, ctx.group, self.H, self.G, self.kd, 0, self.scale, sink=self.sink,
                                       gate=gate)
        return ops.paged_attention_kv(q, ctx.plane, b, ctx.group, self.H, self.G, self.kd, self.vd, ctx.page_size, 0,
                                      self.scale, sink=self.sink, gate=gate)

    def forward32(self, x, ctx):
        return self.ops.linear(self.core(x, ctx), self.w_o, out_dtype=torch.float32)

    def forward(self, x, ctx, residual=None):
        return self.ops.linear(self.core(x, ctx), self.w_o, residual=residual)


@MIXERS.register("latent_attention")
class LatentAttention:
    """Softmax attention whose keys and values are made from one low-rank latent per position.

    q = x.Wq^T, a head being [dim unrotated | rot_dim rotated] channels; with q_rank > 0 the queries go through a latent
    of their own, q = rmsnorm(x.Wdq^T).Wuq^T. x.Wdkv^T gives rank + rot_dim channels: the first rank, RMS-normed with a
    gain, are the latent c; the others are one rotated key part that all heads share. Head h's unrotated key is Wuk[h] c
    and its value Wuv[h] c; score = (q_plain . k_plain + q_rot . k_rot) * scale; rotation of the first rot_dims channels of
    the rotated parts in interleaved pairs (pair_half: in the pairs (i, i + rot_dims / 2)) by position * base^(-2i/rot_dims),
    or by the frequencies and with the factor of `slowed_frequencies` (rot_slowed); causal softmax over all earlier
    positions or the last `window`, with a learned sink per head (sink: one more key of score sink[h], not scaled, without
    a value); the heads side by side are multiplied by sigmoid(x.Wg^T) channel by channel (gate); out = heads . Wo^T.

    Only c and the rotated key part are kept, as one key of rank + rot_dim channels per position whose value is c
    again (transposed, as the attention kernels read values). The products with
    Wuk and Wuv are moved to the query's side of the sums: q_plain . (Wuk[h] c) = (Wuk[h]^T q_plain) . c, so a row's
    query becomes [Wuk[h]^T q_plain | q_rot] against the key [c | k_rot]; and sum_j p_j Wuv[h] c_j = Wuv[h] sum_j p_j c_j,
    so the attention's values are the latents themselves and Wuv[h] is applied to the result.

    params: width, n_heads, dim, rot_dim, value_dim, rank, rot_dims, rot_base, scale, eps, and optionally q_rank (0),
    window (0: all), pair_half, rot_slowed, sink, gate. tensors, stored [out, in]: q (heads*(dim+rot_dim), width), or with
    q_rank dq (q_rank, width), dq_norm (q_rank,), uq (heads*(dim+rot_dim), q_rank); dkv (rank+rot_dim, width), dkv_norm
    (rank,), uk (heads*dim, rank), uv (heads*value_dim, rank), o (width, heads*value_dim), with sink: sink (heads,), with
    gate: gate (heads*value_dim, width).
    """
    graph_safe = True

    @classmethod
    def tensor_shapes(cls, params):
        w, H, D, R, V, C = (params[k] for k in ("width", "n_heads", "dim", "rot_dim", "value_dim", "rank"))
        Q = params.get("q_rank", 0)
        shapes = {"dq": (Q, w), "dq_norm": (Q,), "uq": (H * (D + R), Q)} if Q else {"q": (H * (D + R), w)}
        shapes.update({"dkv": (C + R, w), "dkv_norm": (C,), "uk": (H * D, C), "uv": (H * V, C), "o": (w, H * V)})
        if params.get("sink", False):
            shapes["sink"] = (H,)
        if params.get("gate", False):
            shapes["gate"] = (H * V, w)
        return shapes

    @classmethod
    def cache_need(cls, params):
        return PagedKvNeed(1, params["rank"] + params["rot_dim"], int(params.get("window", 0)), value_dim=params["rank"])

    def __init__(self, spec, tensors, ops):
        from .base import to_gain
        p = spec.params
        self.ops = ops
        self.H, self.D, self.R, self.V, self.C = (int(p[k]) for k in ("n_heads", "dim", "rot_dim", "value_dim", "rank"))
        self.q_rank, self.window = int(p.get("q_rank", 0)), int(p.get("window", 0))
        self.rot_dims, self.pair_half = int(p.get("rot_dims", self.R)), bool(p.get("pair_half", False))
        if self.rot_dims % 2 or self.rot_dims > self.R:
            raise ValueError(f"{self.rot_dims} rotated channels of a part of {self.R}: an even number, at most the part")
        self.scale, self.eps = float(p["scale"]), float(p["eps"])
        self.freqs, self.rot_factor = _rotation(ops, self.rot_dims, float(p.get("rot_base", 10000.0)), p.get("rot_slowed"))
        # one product for everything that reads the row; every block of it starts at a multiple of 8 rows
        mats = [tensors.of(spec, "dq" if self.q_rank else "q"), tensors.of(spec, "dkv")]
        if p.get("gate", False):
            mats.append(tensors.of(spec, "gate"))
        w_in, starts = stacked_rows(mats)
        self.c_at, self.g_at = starts[1], starts[2] if len(mats) > 2 else None
        self.w_in = to_compute(ops, w_in)
        if self.q_rank:
            self.q_gain = to_gain(ops, tensors.of(spec, "dq_norm"))
            self.w_uq = to_compute(ops, tensors.of(spec, "uq"))
        self.sink = to_gain(ops, tensors.of(spec, "sink")) if p.get("sink", False) else None
        self.c_gain = to_gain(ops, tensors.of(spec, "dkv_norm"))
        # [heads, rank, dim]: Wuk[h]^T, which takes a head's unrotated query into the latent's space
        self.w_uk_t = to_compute(ops, tensors.of(spec, "uk").view(self.H, self.D, self.C).transpose(1, 2))
        self.w_uv = to_compute(ops, tensors.of(spec, "uv").view(self.H, self.V, self.C))
        self.w_o = to_compute(ops, tensors.of(spec, "o"))

    # the matrix-core kernel's items, where a step brings portions
    def plan_key(self):
        return ("latent", self.H) if hasattr(self.ops, "plan_latent") else None

    def plan_rows(self, seq_rows, add, mode=None):
        return self.ops.plan_latent(self.H, seq_rows, add)

    def core(self, x, ctx):
        ops, b = self.ops, ctx.batch
        H, D, R, V, C = self.H, self.D, self.R, self.V, self.C
        proj = ops.linear(x, self.w_in, out_dtype=torch.float32)
        queries = proj
        if self.q_rank:
            queries = ops.linear(ops.rmsnorm32(proj[:, :self.q_rank], self.q_gain, self.eps), self.w_uq, out_dtype=torch.float32)
        q, q_plain = ops.latent_prepare(queries, 0, self.c_at, b.positions, b.write_slots[ctx.group], ctx.plane, H, D, R, C,
                                        ctx.page_size, self.c_gain, self.freqs, self.rot_dims, self.eps, ctx.writes_cache,
                                        latent=proj, pair_half=self.pair_half, rot_factor=self.rot_factor)
        ops.heads_linear(q_plain, self.w_uk_t, q, C + R)
        mixed = ops.latent_attention(q, ctx.plane, b, ctx.group, H, C + R, C, ctx.page_size, self.scale, window=self.window,
                                     sink=self.sink)
        gate = proj[:, self.g_at:self.g_at + H * V] if self.g_at is not None else None
        return ops.heads_linear(mixed, self.w_uv, ops.empty(mixed.shape[0], H * V), V, gate=gate)

    def forward32(self, x, ctx):
        return self.ops.linear(self.core(x, ctx), self.w_o, out_dtype=torch.float32)

    def forward(self, x, ctx, residual=None):
        return self.ops.linear(self.core(x, ctx), self.w_o, residual=residual)


@MIXERS.register("convolved_attention")
class ConvolvedAttention:
    """Grouped-query softmax attention whose queries, keys and values pass a short convolution over time, with keys and
    values turned by their position and a learned sink.

    q = x.Wq^T + bq, k = x.Wk^T + bk, v = x.Wv^T + bv; then, channel by channel, y_t = sum_d taps[K-1-d] u_(t-d) over the row
    and the K - 1 rows before it (nothing before a request's first row). The first rot_dims channels of every query and key
    head are rotated in interleaved pairs by position * base^(-2i/rot_dims), or by the frequencies and with the factor of
    `slowed_frequencies` (rot_slowed). Values are turned over all their channels in interleaved pairs by position *
    turn_base^(-2m/value_dim) and cached so; a head's result at position p is turned back by p (turn_base None: values
    are left as they are). score = q.k * scale; causal softmax over all earlier positions or the last `window` with one
    more key of score sink[h], not scaled, without a value; out = heads . Wo^T + bo. Convolution, angles, scores and the
    softmax are 32-bit.

    The pages hold turned keys and values; a state line per request holds the last taps - 1 projected rows [taps - 1,
    heads*key_dim + kv_heads*(key_dim + value_dim)], oldest first.

    params: width, n_heads, n_kv_heads, key_dim, value_dim, taps, scale, rot_dims, rot_base, rot_slowed, turn_base, window.
    tensors, stored [out, in]: q (heads*key_dim, width), k (kv_heads*key_dim, width), v (kv_heads*value_dim, width), q_bias,
    k_bias, v_bias, q_conv, k_conv, v_conv ([channels, taps], the last column weighs the row itself), sink (heads,),
    o (width, heads*value_dim), o_bias (width,).
    """
    graph_safe = True

    @classmethod
    def tensor_shapes(cls, params):
        w, H, G, kd, vd, K = (params[k] for k in ("width", "n_heads", "n_kv_heads", "key_dim", "value_dim", "taps"))
        shapes = {"sink": (H,), "o": (w, H * vd), "o_bias": (w,)}
        for name, channels in (("q", H * kd), ("k", G * kd), ("v", G * vd)):
            shapes.update({name: (channels, w), name + "_bias": (channels,), name + "_conv": (channels, K)})
        return shapes

    @classmethod
    def cache_need(cls, params):
        H, G, kd, vd, K = (params[k] for k in ("n_heads", "n_kv_heads", "key_dim", "value_dim", "taps"))
        pages = PagedKvNeed(G, kd, int(params.get("window", 0)), value_dim=vd)
        floats = (K - 1) * (H * kd + G * (kd + vd))
        return (pages, StateNeed((floats,), "float32")) if floats else pages

    def __init__(self, spec, tensors, ops):
        from .base import to_gain
        p = spec.params
        self.ops = ops
        self.H, self.G, self.kd, self.vd, self.K = (int(p[k]) for k in ("n_heads", "n_kv_heads", "key_dim", "value_dim", "taps"))
        if self.H % self.G:
            raise ValueError(f"{self.H} query heads are not a multiple of {self.G} key/value heads")
        self.scale, self.window = float(p["scale"]), int(p.get("window", 0))
        self.rot_dims = int(p.get("rot_dims", 0))
        if self.rot_dims % 2 or self.rot_dims > self.kd:
            raise ValueError(f"{self.rot_dims} rotated channels of a head of {self.kd}: an even number, at most the head")
        self.freqs, self.rot_factor = _rotation(ops, self.rot_dims, float(p.get("rot_base", 10000.0)), p.get("rot_slowed"))
        turn = p.get("turn_base")
        if turn is not None and self.vd % 2:
            raise ValueError(f"values of {self.vd} channels cannot be turned in pairs")
        self.turn_freqs = _rotary_frequencies(ops, self.vd, float(turn)) if turn is not None else None
        self.w_in = to_compute(ops, torch.cat([tensors.of(spec, k) for k in ("q", "k", "v")], dim=0))
        self.bias = to_gain(ops, torch.cat([tensors.of(spec, k + "_bias") for k in ("q", "k", "v")], dim=0))
        self.taps = to_gain(ops, torch.cat([tensors.of(spec, k + "_conv") for k in ("q", "k", "v")], dim=0))
        self.sink, self.o_bias = to_gain(ops, tensors.of(spec, "sink")), to_gain(ops, tensors.of(spec, "o_bias"))
        self.w_o = to_compute(ops, tensors.of(spec, "o"))
        self.same = self.kd == self.vd        # then the pages have the layout every attention kernel reads

    # the matrix-core kernels' work lists, where keys and values are of one size (see GqaAttention)
    def plan_key(self):
        if not self.same or not hasattr(self.ops, "plan_attention"):
            return None
        return ("attention", self.H, self.G, self.kd, self.window)

    def plan_mode(self, seq_rows):
        mode = getattr(self.ops, "plan_attention_mode", None)
        return mode(seq_rows, self.window) if mode is not None and self.same else None

    def plan_rows(self, seq_rows, add, mode=None):
        return self.ops.plan_attention(self.H, self.G, self.kd, seq_rows, add, mode, self.window)

    def core(self, x, ctx):
        ops, b = self.ops, ctx.batch
        proj = ops.linear(x, self.w_in, out_dtype=torch.float32)
        q, turn = ops.convolved_prepare(proj, self.bias, self.taps, ctx.state, b, b.write_slots[ctx.group], ctx.plane, self.H,
                                        self.G, self.kd, self.vd, ctx.page_size, self.freqs, self.rot_dims, self.rot_factor,
                                        self.turn_freqs, ctx.writes_cache)
        if self.same:
            return ops.paged_attention(q, ctx.plane, b, ctx.group, self.H, self.G, self.kd, self.window, self.scale,
                                       sink=self.sink, turn=turn)
        return ops.paged_attention_kv(q, ctx.plane, b, ctx.group, self.H, self.G, self.kd, self.vd, ctx.page_size, self.window,
                                      self.scale, sink=self.sink, turn=turn)

    def forward_parts(self, x, ctx):
        """(the result without its output bias, 32-bit; the bias): for a block whose sum adds the bias."""
        return self.ops.linear(self.core(x, ctx), self.w_o, out_dtype=torch.float32), self.o_bias

    def forward32(self, x, ctx):
        y, bias = self.forward_parts(x, ctx)
        return y + bias

    def forward(self, x, ctx, residual=None):
        y = self.forward32(x, ctx)
        if residual is not None:
            y = y + residual.to(torch.float32)
        return y.to(self.ops.dtype)


@MIXERS.register("chunked_attention")
class ChunkedAttention:
    """Grouped-query softmax attention inside chunks of positions, with biased projections and keys and values of
    different sizes.

    q = x.Wq^T + bq, k = x.Wk^T + bk, v = x.Wv^T + bv. The whole of a row's queries (all heads side by side) is RMS-normed
    at once with a gain of heads * key_dim entries, and so is the whole of its keys, before rotation. The first rot_dims
    channels of every query and key head are rotated in the pairs (i, i + rot_dims / 2) by position * rot_base^(-2i /
    rot_dims) / rot_factor; the other channels pass. score = q.k * scale. The row at position p sees the keys j <= p
    with floor(j / chunk) = floor(p / chunk): a chunk's edges are multiples of `chunk` in the request, wherever a prompt
    was cut into portions (chunk 0: all j <= p).
    out = softmax-weighted values of all heads . Wo^T + bo. Norms, angles, scores and the softmax are 32-bit.

    params: width, n_heads, n_kv_heads, key_dim, value_dim, scale, eps, rot_dims, rot_base, rot_factor, chunk. tensors,
    stored [out, in]: q (heads*key_dim, width), k (kv_heads*key_dim, width), v (kv_heads*value_dim, width), q_bias,
    k_bias, v_bias, q_norm (heads*key_dim,), k_norm (kv_heads*key_dim,), o (width, heads*value_dim), o_bias (width,).
    """
    graph_safe = True

    @classmethod
    def tensor_shapes(cls, params):
        w, H, G, kd, vd = (params[k] for k in ("width", "n_heads", "n_kv_heads", "key_dim", "value_dim"))
        return {"q": (H * kd, w), "k": (G * kd, w), "v": (G * vd, w), "q_bias": (H * kd,), "k_bias": (G * kd,),
                "v_bias": (G * vd,), "q_norm": (H * kd,), "k_norm": (G * kd,), "o": (w, H * vd), "o_bias": (w,)}

    @classmethod
    def cache_need(cls, params):
        # every key is kept: a chunk's keys are found through the same block table as any others
        return PagedKvNeed(params["n_kv_heads"], params["key_dim"], 0, value_dim=params["value_dim"])

    def __init__(self, spec, tensors, ops):
        from .base import to_gain
        p = spec.params
        self.ops = ops
        self.H, self.G, self.kd, self.vd = int(p["n_heads"]), int(p["n_kv_heads"]), int(p["key_dim"]), int(p["value_dim"])
        if self.H % self.G:
            raise ValueError(f"{self.H} query heads are not a multiple of {self.G} key/value heads")
        self.scale, self.eps, self.chunk = float(p["scale"]), float(p["eps"]), int(p.get("chunk", 0))
        self.rot_dims = int(p.get("rot_dims", 0))
        if self.rot_dims % 2 or self.rot_dims > self.kd or self.chunk < 0:
            raise ValueError(f"{self.rot_dims} rotated channels of a head of {self.kd} (an even number, at most the head), "
                             f"chunks of {self.chunk}")
        factor = float(p.get("rot_factor", 1.0))
        i = torch.arange(self.rot_dims // 2, dtype=torch.float64)
        freqs = float(p.get("rot_base", 10000.0)) ** (-2.0 * i / max(1, self.rot_dims)) / factor
        self.freqs = freqs.to(torch.float32).to(ops.device)
        mats = [tensors.of(spec, k) for k in ("q", "k", "v")]
        self.k_at = mats[0].shape[0]
        self.v_at = self.k_at + mats[1].shape[0]
        self.w_in = to_compute(ops, torch.cat(mats, dim=0))
        self.q_bias, self.k_bias, self.v_bias, self.o_bias = (to_gain(ops, tensors.of(spec, k))
                                                              for k in ("q_bias", "k_bias", "v_bias", "o_bias"))
        self.q_gain, self.k_gain = to_gain(ops, tensors.of(spec, "q_norm")), to_gain(ops, tensors.of(spec, "k_norm"))
        self.w_o = to_compute(ops, tensors.of(spec, "o"))
        self.same = self.kd == self.vd        # then the pages have the layout every attention kernel reads
        self.span = -self.chunk               # how the attention kernels for one size are told of chunks: a negative window

    # the matrix-core kernels' work lists, where keys and values are of one size (see GqaAttention)
    def plan_key(self):
        if not self.same or not hasattr(self.ops, "plan_attention"):
            return None
        return ("attention", self.H, self.G, self.kd, self.span)

    def plan_mode(self, seq_rows):
        mode = getattr(self.ops, "plan_attention_mode", None)
        return mode(seq_rows, self.span) if mode is not None and self.same else None

    def plan_rows(self, seq_rows, add, mode=None):
        return self.ops.plan_attention(self.H, self.G, self.kd, seq_rows, add, mode, self.span)

    def core(self, x, ctx):
        ops, b = self.ops, ctx.batch
        proj = ops.linear(x, self.w_in, out_dtype=torch.float32)
        q = ops.attention_prepare(proj, 0, self.k_at, self.v_at, b.positions, b.write_slots[ctx.group], ctx.plane, self.H,
                                  self.G, self.kd, self.vd, ctx.page_size, q_gain=self.q_gain, k_gain=self.k_gain,
                                  freqs=self.freqs, rot_dims=self.rot_dims, eps=self.eps, write_cache=ctx.writes_cache,
                                  value_norm=False, q_bias=self.q_bias, k_bias=self.k_bias, v_bias=self.v_bias,
                                  whole_norm=True, pair_half=True)
        if self.same:
            return ops.paged_attention(q, ctx.plane, b, ctx.group, self.H, self.G, self.kd, self.span, self.scale)
        return ops.paged_attention_kv(q, ctx.plane, b, ctx.group, self.H, self.G, self.kd, self.vd, ctx.page_size, 0,
                                      self.scale, chunk=self.chunk)

    def forward_parts(self, x, ctx):
        """(the result without its output bias, 32-bit; the bias): for a block whose sum adds the bias."""
        return self.ops.linear(self.core(x, ctx), self.w_o, out_dtype=torch.float32), self.o_bias

    def forward32(self, x, ctx):
        y, bias = self.forward_parts(x, ctx)
        return y + bias

    def forward(self, x, ctx, residual=None):
        y = self.forward32(x, ctx)
        if residual is not None:
            y = y + residual.to(torch.float32)
        return y.to(self.ops.dtype)


@MIXERS.register("sigmoid_mixed_attention")
class SigmoidMixedAttention:
    """Grouped-query attention inside chunks of positions whose weights are sigmoids, not a softmax, and are mixed across
    the heads before they meet the values.

    q = x.Wq^T + bq, k = x.Wk^T + bk, v = x.Wv^T + bv. The first rot_dims channels of every query and key head are
    rotated in the pairs (i, i + rot_dims / 2) by position * f_i (f from `banded_frequencies`); the other channels pass.
    s = q.k * scale, then s <- softcap * tanh(s / softcap) (softcap 0: as it is). The row at position p sees the keys
    j <= p with floor(j / chunk) = floor(p / chunk) (chunk 0: all j <= p); a seen key's weight for head g is
    w_g = sigmoid(s + head_bias[g]), each key on its own. Head h then uses sum_g talk[h, g] * w_g on the values of its
    own key/value head; out = heads . Wo^T. Angles, scores and weights are 32-bit.

    params: width, n_heads, n_kv_heads, key_dim, value_dim, scale, softcap, chunk, rot_dims, rot_base, rot_bands
    ((factor, low, high, original) or None). tensors, stored [out, in]: q (heads*key_dim, width), k (kv_heads*key_dim,
    width), v (kv_heads*value_dim, width), q_bias, k_bias, v_bias, head_bias (heads,), talk (heads, heads),
    o (width, heads*value_dim).
    """
    graph_safe = True

    @classmethod
    def tensor_shapes(cls, params):
        w, H, G, kd, vd = (params[k] for k in ("width", "n_heads", "n_kv_heads", "key_dim", "value_dim"))
        return {"q": (H * kd, w), "k": (G * kd, w), "v": (G * vd, w), "q_bias": (H * kd,), "k_bias": (G * kd,),
                "v_bias": (G * vd,), "head_bias": (H,), "talk": (H, H), "o": (w, H * vd)}

    @classmethod
    def cache_need(cls, params):
        # every key is kept: a chunk's keys are found through the same block table as any others
        return PagedKvNeed(params["n_kv_heads"], params["key_dim"], 0, value_dim=params["value_dim"])

    def __init__(self, spec, tensors, ops):
        from .base import to_gain
        p = spec.params
        self.ops = ops
        self.H, self.G, self.kd, self.vd = int(p["n_heads"]), int(p["n_kv_heads"]), int(p["key_dim"]), int(p["value_dim"])
        if self.H % self.G:
            raise ValueError(f"{self.H} query heads are not a multiple of {self.G} key/value heads")
        self.scale, self.softcap, self.chunk = float(p["scale"]), float(p.get("softcap", 0.0)), int(p.get("chunk", 0))
        self.rot_dims = int(p.get("rot_dims", 0))
        if self.rot_dims % 2 or self.rot_dims > self.kd or self.chunk < 0 or self.softcap < 0:
            raise ValueError(f"{self.rot_dims} rotated channels of a head of {self.kd} (an even number, at most the head), "
                             f"chunks of {self.chunk}, a cap of {self.softcap}")
        self.freqs = _rotary_frequencies(ops, self.rot_dims, float(p.get("rot_base", 10000.0)), p.get("rot_bands"))
        mats = [tensors.of(spec, k) for k in ("q", "k", "v")]
        self.input_rows = torch.cat(mats, dim=0)        # as stored: a block may fuse them into a wider product
        self.k_at = mats[0].shape[0]
        self.v_at = self.k_at + mats[1].shape[0]
        self._w_in = None
        self.q_bias, self.k_bias, self.v_bias = (to_gain(ops, tensors.of(spec, k)) for k in ("q_bias", "k_bias", "v_bias"))
        self.head_bias = to_gain(ops, tensors.of(spec, "head_bias"))
        self.talk = to_gain(ops, tensors.of(spec, "talk"))
        self.w_o = to_compute(ops, tensors.of(spec, "o"))

    # the matrix-core kernel's items (tiles of up to 16 rows of one request), where a step brings portions
    def plan_key(self):
        return ("row_tiles", 16) if hasattr(self.ops, "plan_row_tiles") else None

    def plan_rows(self, seq_rows, add, mode=None):
        return self.ops.plan_row_tiles(seq_rows, add)

    def core(self, proj, ctx):
        ops, b = self.ops, ctx.batch
        q = ops.attention_prepare(proj, 0, self.k_at, self.v_at, b.positions, b.write_slots[ctx.group], ctx.plane, self.H,
                                  self.G, self.kd, self.vd, ctx.page_size, freqs=self.freqs, rot_dims=self.rot_dims,
                                  write_cache=ctx.writes_cache, value_norm=False, q_bias=self.q_bias, k_bias=self.k_bias,
                                  v_bias=self.v_bias, pair_half=True)
        return ops.mixed_sigmoid_attention(q, ctx.plane, b, ctx.group, self.H, self.G, self.kd, self.vd, ctx.page_size,
                                           self.chunk, self.scale, self.softcap, self.head_bias, self.talk)

    def forward_projected(self, proj, ctx):
        """From this mixer's columns of a 32-bit input product to its result in 32-bit."""
        return self.ops.linear(self.core(proj, ctx), self.w_o, out_dtype=torch.float32)

    def forward32(self, x, ctx):
        if self._w_in is None:
            self._w_in = to_compute(self.ops, self.input_rows)
        return self.forward_projected(self.ops.linear(x, self._w_in, out_dtype=torch.float32), ctx)

    def forward(self, x, ctx, residual=None):
        y = self.forward32(x, ctx)
        if residual is not None:
            y = y + residual.to(torch.float32)
        return y.to(self.ops.dtype)


@MIXERS.register("capped_attention")
class CappedAttention:
    """Causal grouped-query softmax attention with capped scores over queries and keys of unit length, keys and values of
    different sizes, and a gate per output channel.

    q = x.Wq^T + bq, k = x.Wk^T + bk, v = x.Wv^T + bv. The first rot_dims channels of every query and key head are rotated
    in the pairs (i, i + rot_dims / 2) by position * rot_base^(-2i/rot_dims), or by the frequencies and with the factor of
    `slowed_frequencies` (rot_slowed); the other channels pass. Then every query and key head is divided by its root mean
    square (unit_qk; eps under the root, no gain). s = q.k * scale, s <- softcap * tanh(s / softcap) (softcap 0: as it is);
    causal softmax over all earlier positions; the heads side by side are multiplied by sigmoid(x.Wg^T) channel by
    channel (gate); out = heads . Wo^T. Angles, norms, scores, the softmax and the gate's sigmoid are 32-bit.

    params: width, n_heads, n_kv_heads, key_dim, value_dim, scale, softcap (0), eps, rot_dims (0), rot_base, rot_slowed
    ((factor, original, fast, slow) or None), unit_qk (true), gate (true). tensors, stored [out, in]: q (heads*key_dim,
    width), k (kv_heads*key_dim, width), v (kv_heads*value_dim, width), q_bias, k_bias, v_bias, with gate: gate
    (heads*value_dim, width), o (width, heads*value_dim).
    """
    graph_safe = True

    @classmethod
    def tensor_shapes(cls, params):
        w, H, G, kd, vd = (params[k] for k in ("width", "n_heads", "n_kv_heads", "key_dim", "value_dim"))
        shapes = {"q": (H * kd, w), "k": (G * kd, w), "v": (G * vd, w), "q_bias": (H * kd,), "k_bias": (G * kd,),
                  "v_bias": (G * vd,), "o": (w, H * vd)}
        if params.get("gate", True):
            shapes["gate"] = (H * vd, w)
        return shapes

    @classmethod
    def cache_need(cls, params):
        return PagedKvNeed(params["n_kv_heads"], params["key_dim"], 0, value_dim=params["value_dim"])

    def __init__(self, spec, tensors, ops):
        from .base import to_gain
        p = spec.params
        self.ops = ops
        self.H, self.G, self.kd, self.vd = int(p["n_heads"]), int(p["n_kv_heads"]), int(p["key_dim"]), int(p["value_dim"])
        if self.H % self.G:
            raise ValueError(f"{self.H} query heads are not a multiple of {self.G} key/value heads")
        self.scale, self.softcap, self.eps = float(p["scale"]), float(p.get("softcap", 0.0)), float(p["eps"])
        self.rot_dims, self.unit_qk = int(p.get("rot_dims", 0)), bool(p.get("unit_qk", True))
        if self.rot_dims % 2 or self.rot_dims > self.kd or self.softcap < 0:
            raise ValueError(f"{self.rot_dims} rotated channels of a head of {self.kd} (an even number, at most the head), a cap "
                             f"of {self.softcap}")
        self.freqs, self.rot_factor = _rotation(ops, self.rot_dims, float(p.get("rot_base", 10000.0)), p.get("rot_slowed"))
        mats = [tensors.of(spec, k) for k in ("q", "k", "v")] + ([tensors.of(spec, "gate")] if p.get("gate", True) else [])
        # one product for everything that reads the row; every block of it starts at a multiple of 8 rows
        w_in, starts = stacked_rows(mats)
        self.k_at, self.v_at, self.g_at = starts[1], starts[2], starts[3] if len(mats) > 3 else None
        self.w_in = to_compute(ops, w_in)
        self.q_bias, self.k_bias, self.v_bias = (to_gain(ops, tensors.of(spec, k)) for k in ("q_bias", "k_bias", "v_bias"))
        self.w_o = to_compute(ops, tensors.of(spec, "o"))

    # the matrix-core kernels' work lists (see GqaAttention)
    def plan_key(self):
        return ("attention", self.H, self.G, max(self.kd, self.vd), 0) if hasattr(self.ops, "plan_attention") else None

    def plan_mode(self, seq_rows):
        mode = getattr(self.ops, "plan_attention_mode", None)
        return mode(seq_rows, 0) if mode is not None else None

    def plan_rows(self, seq_rows, add, mode=None):
        return self.ops.plan_attention(self.H, self.G, max(self.kd, self.vd), seq_rows, add, mode, 0)

    def core(self, x, ctx):
        ops, b = self.ops, ctx.batch
        proj = ops.linear(x, self.w_in, out_dtype=torch.float32)
        q = ops.attention_prepare(proj, 0, self.k_at, self.v_at, b.positions, b.write_slots[ctx.group], ctx.plane, self.H,
                                  self.G, self.kd, self.vd, ctx.page_size, freqs=self.freqs, rot_dims=self.rot_dims,
                                  eps=self.eps, write_cache=ctx.writes_cache, value_norm=False, q_bias=self.q_bias,
                                  k_bias=self.k_bias, v_bias=self.v_bias, pair_half=True, rot_factor=self.rot_factor,
                                  unit_rms=self.unit_qk)
        gate = proj[:, self.g_at:self.g_at + self.H * self.vd] if self.g_at is not None else None
        return ops.paged_attention_kv(q, ctx.plane, b, ctx.group, self.H, self.G, self.kd, self.vd, ctx.page_size, 0, self.scale,
                                      softcap=self.softcap, channel_gate=gate, matrix_cores=True)

    def forward32(self, x, ctx):
        return self.ops.linear(self.core(x, ctx), self.w_o, out_dtype=torch.float32)

    def forward(self, x, ctx, residual=None):
        return self.ops.linear(self.core(x, ctx), self.w_o, residual=residual)
