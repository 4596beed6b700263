"""Parts around a stream to which a sublayer's normed output is added: the block ``h <- h + m norm(sublayer(h))`` with a
short convolution over time ahead of its mixer, the norm with one number for all channels, attention whose heads are
the difference of two maps, linear attention whose forget gate also says what is written, and the gated feed-forward
with an activation by name.

Kinds registered here: norm ``rmsnorm_scalar``; input_conv ``causal``; mixer ``differential_attention`` and
``forget_memory``; feed_forward ``gated_mlp``; block ``added_norm``.  Every size and constant is a parameter of the
part's spec.
"""
from __future__ import annotations

import math
from dataclasses import dataclass, replace
from typing import Optional

import torch

from .. import kernels as K
from ..registry import register_part
from .base import Block, CacheNeed, KVNeed, LayerCache, Part, StateNeed, WeightRequest
from .hybrid import PagedSoftmax
from .postnorm import StreamCopy
from .standard import RMSNorm, SwiGLU, build_part, requests_of


def _up4(n: int) -> int:
    return (n + 3) // 4 * 4


# ------------------------------------------------------------------ norm

@register_part("norm", "rmsnorm_scalar")
class ScalarRMSNorm(RMSNorm):
    """``x * rsqrt(mean(x^2) + eps) * g`` in float32 with one number g for all channels.  params: size, eps.
    weights: weight [] (a tensor without dimensions).  The device holds g once a channel, so the kernels of norms with
    a weight a channel serve it."""

    @classmethod
    def weight_requests(cls, spec):
        return [WeightRequest(spec.weights["weight"], ())]

    def __init__(self, spec, weights, rt):
        row = weights["weight"].to(torch.float32).reshape(1).expand(int(spec.params["size"]))
        super().__init__(spec, {"weight": row}, rt)


# ------------------------------------------------------------------ a sublayer's input, convolved over time

@register_part("input_conv", "causal")
class CausalInputConv(Part):
    """``x[t] = h[t] + sum_j W[:, j] * h[t - (taps - 1 - j)]``, every channel by itself, zeros before a sequence's first
    token.  The last ``taps - 1`` rows h of a sequence are kept, in float32, in the block's per-request state.
    params: size, taps.  weights: filters [size, taps]."""

    graph_safe = True
    idempotent = False        # a step moves the kept rows on

    @classmethod
    def weight_requests(cls, spec):
        return [WeightRequest(spec.weights["filters"], (spec.params["size"], spec.params["taps"]))]

    def __init__(self, spec, weights, rt):
        super().__init__(spec, weights, rt)
        self.size, self.taps = int(spec.params["size"]), int(spec.params["taps"])
        self.filters = weights["filters"].to(device=rt.device, dtype=torch.float32).contiguous()
        self.state_floats = (self.taps - 1) * self.size
        K.short_conv_lib()


# ------------------------------------------------------------------ attention as the difference of two maps

@register_part("mixer", "differential_attention")
class DifferentialAttention(Part):
    """Causal softmax attention with grouped heads, each of two maps: two query and key vectors of ``key_dim`` and one
    value.  The projected queries, keys and values pass a causal convolution over ``taps`` tokens a channel (None: none);
    every query and key vector is normed with one weight shared by heads and maps and rotated (``position``: neighbouring
    channel pairs; None: not), in float32.  ``score = q . k * scale``, then ``softcap tanh(score / softcap)`` (None: not);
    query i sees key j <= i in its own chunk of ``chunk`` positions, counted from the sequence's first (None: all).  With
    a1, a2 the maps' outputs over the head's values, ``o = a1 - lambda a2`` is divided by its root mean square over the
    value channels and multiplied by ``1 - diff``; then ``W_o``.  ``lambda = exp(lq1 . lk1) - exp(lq2 . lk2) + diff``, one
    number, is worked out once, at load.

    A token keeps both maps' keys side by side and one value in the pages; of a chunked attention the pages of the last
    ``chunk`` keys.  The last ``taps - 1`` projected rows are the per-request state.

    params: hidden_size, num_heads, num_kv_heads, key_dim, value_dim, scale, softcap, chunk, taps, diff, eps, position.
    weights: q [H*2*dk, d], k [G*2*dk, d], v [G*dv, d], o [d, H*dv], q_norm, k_norm, lq1, lk1, lq2, lk2 [dk]; with taps also
    q_conv [H*2*dk, taps], k_conv [G*2*dk, taps], v_conv [G*dv, taps]."""

    graph_safe = True
    MAPS = 2

    @classmethod
    def weight_requests(cls, spec):
        p, w = spec.params, spec.weights
        d, H, G, dk, dv, m = p["hidden_size"], p["num_heads"], p["num_kv_heads"], p["key_dim"], p["value_dim"], cls.MAPS
        rows = {"q": H * m * dk, "k": G * m * dk, "v": G * dv}
        out = [WeightRequest(w[k], (n, d)) for k, n in rows.items()] + [WeightRequest(w["o"], (d, H * dv))]
        out += [WeightRequest(w[k], (dk,)) for k in ("q_norm", "k_norm", "lq1", "lk1", "lq2", "lk2")]
        if p.get("taps") is not None:
            out += [WeightRequest(w[f"{k}_conv"], (n, p["taps"])) for k, n in rows.items()]
        if p.get("position") is not None:
            out += requests_of("position", p["position"])
        return out

    def __init__(self, spec, weights, rt):
        super().__init__(spec, weights, rt)
        p, names = spec.params, spec.weights
        self.H, self.G, self.dk, self.dv = (int(p[k]) for k in ("num_heads", "num_kv_heads", "key_dim", "value_dim"))
        self.eps, self.diff = float(p["eps"]), float(p["diff"])
        self.chunk = None if p.get("chunk") is None else int(p["chunk"])
        self.taps = 1 if p.get("taps") is None else int(p["taps"])
        self.idempotent = self.taps < 2           # with a convolution a step moves the kept rows on
        self.core = PagedSoftmax(self.H * self.MAPS, self.G * self.MAPS, self.dk, self.dv, float(p["scale"]), softcap=p.get("softcap"),
                                 chunk=self.chunk, maps=self.MAPS)
        order = ("q", "k", "v")
        self.w_qkv = rt.weight("|".join(names[k] for k in order), torch.cat([weights[k] for k in order], dim=0))
        self.w_o = rt.weight(names["o"], weights["o"])
        self.q_norm, self.k_norm = (rt.vector32(names[k], weights[k]) for k in ("q_norm", "k_norm"))
        self.filters = None
        if p.get("taps") is not None:
            self.filters = torch.cat([weights[f"{k}_conv"] for k in order], dim=0).to(device=rt.device, dtype=torch.float32).contiguous()
        self.freq = None
        if p.get("position") is not None:
            self.freq, amplitude = build_part("position", p["position"], getattr(weights, "checkpoint", {}), rt).frequencies()
            if amplitude != 1.0 or 2 * self.freq.shape[0] > self.dk:
                raise ValueError(f"{2 * self.freq.shape[0]} channels rotated with amplitude {amplitude} do not fit this part")
        l = {k: weights[k].to(torch.float64) for k in ("lq1", "lk1", "lq2", "lk2")}
        self.factor = math.exp(float((l["lq1"] * l["lk1"]).sum())) - math.exp(float((l["lq2"] * l["lk2"]).sum())) + self.diff
        self.channels = int(self.w_qkv.shape[0])
        self.state_floats = (self.taps - 1) * self.channels
        K.short_conv_lib()

    def cache_need(self) -> CacheNeed:
        state = StateNeed((_up4(self.state_floats),), torch.float32) if self.state_floats else None
        return CacheNeed(kv=KVNeed(self.G, self.MAPS * self.dk, self.chunk, self.dv), state=state)

    def forward(self, x, ctx, cache: LayerCache, out: Optional[torch.Tensor] = None):
        if not cache.writes:
            raise K.KernelError("a differential_attention part writes the keys and values it makes")
        T = x.shape[0]
        proj = K.linear(x, self.w_qkv, out_dtype=torch.float32)
        q = torch.empty(T, self.H * self.MAPS * self.dk, dtype=self.rt.dtype, device=x.device)
        K.qkv_conv(proj, ctx.positions, cache.slot_mapping, self.filters, self.q_norm, self.k_norm, self.eps, self.freq, cache.state, 0, ctx,
                   q, cache.kpool, cache.vpool, self.H, self.MAPS)
        rows, runs = self.core.unfinished(q, ctx, cache.kpool, cache.vpool, cache.block_table)
        y = torch.empty(T, self.H * self.dv, dtype=self.rt.dtype, device=x.device)
        K.merge_maps(rows, T, self.H, self.G, self.dv, runs, self.factor, self.eps, 1.0 - self.diff, y)
        return K.linear(y, self.w_o, out_dtype=torch.float32, out=out)


# ------------------------------------------------------------------ linear attention, a gate that forgets and writes

@register_part("mixer", "forget_memory")
class ForgetMemory(Part):
    """Linear attention with one forget gate a head and key channel that also says how much of the value is written.  Per
    head, with a memory ``S`` [key channel, value channel] in float32 that starts at zero and is carried from token to token:

        ``f = l + (1 - l) sigmoid(W_f x + b);  S <- diag(f) S + (1 - f) v^T;  o = S^T silu(W_q x)``          v = W_v x

    Every head's read-out is divided by its root mean square and multiplied by ``norm``, one weight shared by the heads; then
    ``W_o``.  The memory is the per-request state.

    params: hidden_size, num_heads, key_dim, value_dim, eps.
    weights: q, f [H*dk, d], f_b, lower [H*dk], v [H*dv, d], norm [dv], o [d, H*dv]."""

    graph_safe = True
    idempotent = False        # a step moves the memory on

    @classmethod
    def weight_requests(cls, spec):
        p, w = spec.params, spec.weights
        d, H, dk, dv = p["hidden_size"], p["num_heads"], p["key_dim"], p["value_dim"]
        return [WeightRequest(w["q"], (H * dk, d)), WeightRequest(w["f"], (H * dk, d)), WeightRequest(w["f_b"], (H * dk,)),
                WeightRequest(w["lower"], (H * dk,)), WeightRequest(w["v"], (H * dv, d)), WeightRequest(w["norm"], (dv,)),
                WeightRequest(w["o"], (d, H * dv))]

    def __init__(self, spec, weights, rt):
        super().__init__(spec, weights, rt)
        p, names = spec.params, spec.weights
        self.H, self.dk, self.dv, self.eps = int(p["num_heads"]), int(p["key_dim"]), int(p["value_dim"]), float(p["eps"])
        order = ("q", "f", "v")
        self.w_in = rt.weight("|".join(names[k] for k in order), torch.cat([weights[k] for k in order], dim=0))
        self.w_o = rt.weight(names["o"], weights["o"])
        self.f_b, self.lower, self.norm = (rt.vector32(names[k], weights[k]) for k in ("f_b", "lower", "norm"))
        self.state_floats = K.forget_state_floats(self.H, self.dk, self.dv)
        K.forget_memory_lib()

    def cache_need(self) -> CacheNeed:
        return CacheNeed(state=StateNeed((self.state_floats,), torch.float32))

    def forward(self, x, ctx, cache: LayerCache, out: Optional[torch.Tensor] = None):
        if not cache.writes:
            raise K.KernelError("a forget_memory mixer moves its memory on: it cannot read another entry's cache")
        seq = ctx.per_seq
        proj = K.linear(x, self.w_in, out_dtype=torch.float32)      # float32 out: everything here enters the recurrence
        o = K.forget_memory(proj, self.f_b, self.lower, cache.state, seq.q_start, seq.q_len, seq.state_slot, self.H, self.dk, self.dv,
                            max_q_len=ctx.max_q_len)
        return K.linear(K.head_norm(o, self.norm, self.eps, self.rt.dtype), self.w_o, out_dtype=torch.float32, out=out)


# ------------------------------------------------------------------ feed-forward

@register_part("feed_forward", "gated_mlp")
class GatedMLP(SwiGLU):
    """``W_down (act(W_gate x) * (W_up x))`` with the activation by name (``activation``: one of
    ``kernels.GATED_ACTIVATIONS``), its result in float32.  params: hidden_size, intermediate_size, activation.
    weights: gate [I, d], up [I, d], down [d, I]."""

    def __init__(self, spec, weights, rt):
        super().__init__(spec, weights, rt)
        self.activation = str(spec.params.get("activation", "silu"))
        if self.activation not in K.GATED_ACTIVATIONS:
            raise ValueError(f"activation {self.activation!r} is not one of {sorted(K.GATED_ACTIVATIONS)}")

    # its products are given a plain input and leave the stream alone
    def takes_normed(self, T: int) -> bool:
        return False

    def takes_scaled(self, T: int) -> bool:
        return False

    def adds_residual(self, T: int) -> bool:
        return False

    def leaves_scaled(self, T: int) -> bool:
        return False

    def carries_addends(self, T: int, addends: int) -> bool:
        return False

    def takes_halved(self, T: int) -> bool:
        cls = type(self)
        return (cls.forward is GatedMLP.forward and cls.hidden is GatedMLP.hidden
                and K.takes_halved(T, self.w_gate_up.shape[1], self.rt.dtype, self.w_gate_up))

    def hidden(self, x) -> torch.Tensor:
        return K.linear_swiglu(x, self.w_gate_up, self.activation)

    def forward(self, x, ctx):
        return K.linear(self.hidden(x), self.w_down, out_dtype=torch.float32)


# ------------------------------------------------------------------ block

@dataclass
class DeferredSum:
    """What an ``added_norm`` block hands on as ``pending`` to a block that ``takes_deferred``: the stream has not received
    ``mult * norm(y)``; the block behind adds it together with what it does to the stream first."""

    y: torch.Tensor
    norm: object
    mult: float

    def add_to(self, h: torch.Tensor, x: Optional[torch.Tensor] = None, conv: Optional["K.InputConv"] = None) -> torch.Tensor:
        return K.add_norm(h, self.y, self.norm.weight, self.mult, self.norm.eps, x=x, conv=conv)


@register_part("block", "added_norm")
class AddedNormBlock(Block):
    """``h += mult * norm1(mixer(conv(h))); h += mult * norm2(ffn(h))``: the sublayers read the stream itself (the mixer
    through ``mixer_conv``, where the block has one), their float32 outputs are normed before they are added to the float32
    stream.  ``ffn`` and ``ffn_norm`` may be absent together, ``mixer_conv`` alone.  The convolution's rows are kept behind
    the mixer's state in the same row of the state slots.  params: mult."""

    ROLES = {"mixer_conv": "input_conv", "mixer": "mixer", "mixer_norm": "norm", "ffn": "feed_forward", "ffn_norm": "norm"}
    OPTIONAL = ("mixer_conv", "ffn", "ffn_norm")
    takes_deferred = defers_sum = True      # ``forward`` takes ``defer=``: its last sum may be left to the block behind

    @classmethod
    def _roles(cls, spec):
        missing = [r for r in cls.ROLES if r not in spec.parts and r not in cls.OPTIONAL]
        extra = [r for r in spec.parts if r not in cls.ROLES]
        if ("ffn" in spec.parts) != ("ffn_norm" in spec.parts):
            missing.append("ffn_norm" if "ffn" in spec.parts else "ffn")
        if missing or extra:
            raise ValueError(f"a block of kind {spec.kind!r} has the parts {sorted(cls.ROLES)}; "
                             f"missing: {missing}, not known: {extra}")
        return [(r, f) for r, f in cls.ROLES.items() if r in spec.parts]

    def __init__(self, spec, tensors, rt):
        super().__init__(spec, tensors, rt)
        self.mult = float(spec.params.get("mult", 1.0))
        self._lay_out_state()
        K.short_conv_lib()

    def _lay_out_state(self) -> None:
        """A request's row of state: the mixer's floats, then (from ``conv_off`` on) the rows of the input's convolution."""
        need = self.mixer.cache_need()
        if need.state is not None and (need.state.dtype != torch.float32 or len(need.state.shape) != 1):
            raise ValueError("an added_norm block's mixer keeps a row of float32 per request, or nothing")
        mixer_floats = 0 if need.state is None else int(need.state.shape[0])
        self.conv_off = _up4(mixer_floats)
        conv_floats = self.mixer_conv.state_floats if "mixer_conv" in self.roles else 0
        floats = self.conv_off + _up4(conv_floats)
        # (a convolution of one tap keeps nothing, but its kernel is handed a state all the same)
        if "mixer_conv" in self.roles:
            floats = max(floats, 4)
        self._need = replace(need, state=StateNeed((floats,), torch.float32) if floats else None)

    def cache_need(self) -> CacheNeed:
        return self._need

    def _sum(self, y, norm) -> DeferredSum:
        return DeferredSum((y if y.dtype == torch.float32 else y.to(torch.float32)).contiguous(), norm, self.mult)

    def _compute_copy(self, h):
        """Where a norm's kernel is to leave the stream in the compute type (None: the stream is in that type itself)."""
        return None if self.rt.dtype == torch.float32 else torch.empty(h.shape, dtype=self.rt.dtype, device=h.device)

    def _mixer_input(self, h, pending, ctx, cache: LayerCache):
        if "mixer_conv" not in self.roles:
            if isinstance(pending, StreamCopy):
                return pending.x
            x = self._compute_copy(h)
            if pending is not None:
                pending.add_to(h, x)
            elif x is not None:
                x.copy_(h)
            return h if x is None else x
        conv = K.InputConv(self.mixer_conv.filters, cache.state, self.conv_off, ctx)
        x = torch.empty(h.shape, dtype=self.rt.dtype, device=h.device)
        if isinstance(pending, DeferredSum):
            if conv.single(h.shape[0]) and h.shape[1] <= K.add_norm_max():
                pending.add_to(h, x, conv)
                return x
            pending.add_to(h)
        return K.input_conv(h, conv, x)

    def forward(self, h, pending, ctx, cache: LayerCache, defer: bool = False):
        if pending is not None and not isinstance(pending, (DeferredSum, StreamCopy)):
            raise K.KernelError("an added_norm block reads a complete stream, or one that lacks a normed sum")
        x = self._mixer_input(h, pending, ctx, cache)
        last = self._sum(self.mixer.forward(x, ctx, cache), self.mixer_norm)
        if "ffn" in self.roles:
            x = self._compute_copy(h)
            last.add_to(h, x)
            last = self._sum(self.ffn.forward(h if x is None else x, ctx), self.ffn_norm)
        if defer:
            return h, last
        last.add_to(h)
        return h, None
