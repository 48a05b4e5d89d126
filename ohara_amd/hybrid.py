"""Building blocks of hybrid decoders (attention layers beside recurrent ones) over the HIP kernels.

Every class is one mechanism with its sizes and constants as constructor arguments; none knows a model's
config keys or tensor names.  A mixer offers ``state(rows, max_seq_length)`` (the tensors it keeps per sequence) and
``__call__(h, state, seq)`` with h the (rows, width rounded up to 8) activations of the call and ``seq`` an
``ops.Seq``.  Mixers that can stand side by side in a ``ParallelMixer`` also offer ``heads_of(p, state, seq, out)``, what they do
between their input projections (rows of p) and their output projection.  Activations, caches and matrices are bfloat16 or, for a model served in 32-bit, fp32; the residual
stream, norms, scores, decays and recurrent states are fp32 in both.
"""

from __future__ import annotations

import ctypes
import math
from dataclasses import dataclass

import torch
import torch.nn.functional as F

from . import ops
from ._lib import DELTA_SILU_GATE, RETENTION_CHUNK, ROUTER_PLAIN, ROUTER_SIGMOID, OharaDelta, OharaGlu, OharaRetention, check, lib

BF16, F32 = torch.bfloat16, torch.float32


def _pad(w: torch.Tensor, rows: int, cols: int | None = None) -> torch.Tensor:
    """Zero rows / columns up to the given sizes."""
    if w.ndim == 1:
        return F.pad(w, (0, rows - w.shape[0]))
    return F.pad(w, (0, (cols or w.shape[1]) - w.shape[1], 0, rows - w.shape[0]))


class Linear:
    """y = x W^T (+ bias).  Inputs and outputs are padded to multiples of 8 columns (the pad rows and columns of W are
    zero, so an output's pad columns are exact zeros); ``exact`` keeps W's own row count.  ``cap``: the result is
    soft-capped, cap * tanh(y / cap)."""

    def __init__(self, w: torch.Tensor, bias: torch.Tensor | None = None, *, dtype=BF16, device="cuda", exact: bool = False,
                 cap: float = 0.0):
        n, k = w.shape
        self.n, self.k, self.dtype, self.cap = (n if exact else ops.round8(n)), ops.round8(k), dtype, float(cap)
        w = _pad(w.detach().to(device=device, dtype=dtype), self.n, self.k).contiguous()
        self.bias = None if bias is None else _pad(bias.detach().to(device=device, dtype=dtype), self.n).contiguous()
        self.w = w if dtype == F32 else ops.pack_linear(w)

    def __call__(self, x: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
        if self.dtype == F32:
            return ops.gemm_f32(x, self.w, self.bias, cap=self.cap, out=out)
        if self.cap:
            return ops.gemm_softcap(x, self.w, self.cap, out=out)
        if self.bias is not None:
            return ops.linear_bias(x, self.w, self.bias, out=out)
        if x.stride(0) != x.shape[1]:
            return ops.gemm(x, self.w, out=out)  # a column slice of a wider buffer
        return ops.gemm_skinny(x, self.w, out=out)

    def tensors(self):
        yield self.w if self.dtype == F32 else self.w.data
        if self.bias is not None:
            yield self.bias


class SwiGLU:
    """down(silu(gate x) * (up x)); gate and up are one launch."""

    def __init__(self, gate, up, down, *, dtype=BF16, device="cuda"):
        ff, k = gate.shape
        ffp, kp = ops.round8(ff), ops.round8(k)
        gate, up = (_pad(w.detach().to(device=device, dtype=dtype), ffp, kp).contiguous() for w in (gate, up))
        self.dtype = dtype
        self.gate_up = (gate, up) if dtype == F32 else ops.pack_gate_up(gate, up)
        self.down = Linear(_pad(down.detach(), down.shape[0], ffp), dtype=dtype, device=device)

    def __call__(self, x: torch.Tensor) -> torch.Tensor:
        if self.dtype == F32:
            act = ops.gemm_f32(x, self.gate_up[0], w_up=self.gate_up[1])
        else:
            act = ops.gemm_skinny(x, self.gate_up)
        return self.down(act)

    def tensors(self):
        yield from (self.gate_up if self.dtype == F32 else (self.gate_up.data,))
        yield from self.down.tensors()


class ClampedGLU:
    """down(g sigmoid(alpha g) (u + offset)), g = gate x capped by ``limit`` from above, u = up x from both sides; gate and up are one
    launch."""

    def __init__(self, gate, up, down, *, limit: float, alpha: float = 1.702, offset: float = 1.0, dtype=BF16, device="cuda"):
        ff, k = gate.shape
        ffp, kp = ops.round8(ff), ops.round8(k)
        gate, up = (_pad(w.detach().to(device=device, dtype=dtype), ffp, kp).contiguous() for w in (gate, up))
        self.dtype, self.ff = dtype, ffp
        self.constants = (float(limit), float(alpha), float(offset))
        self.gate_up = (gate, up) if dtype == F32 else ops.pack_gate_up(gate, up)
        self.down = Linear(_pad(down.detach(), down.shape[0], ffp), dtype=dtype, device=device)

    def __call__(self, x: torch.Tensor) -> torch.Tensor:
        return self.down(ops.gemm_glu(x, self.gate_up, *self.constants))

    def tensors(self):
        yield from (self.gate_up if self.dtype == F32 else (self.gate_up.data,))
        yield from self.down.tensors()


class XieluMLP:
    """down(f(up x + up_bias)) + down_bias, f(z) = z / 2 + (softplus(p) z^2 if z > 0 else (1/2 + softplus(q)) (exp(z) - 1 - z))."""

    def __init__(self, up, up_bias, down, down_bias, p: float, q: float, *, dtype=BF16, device="cuda"):
        softplus = lambda v: F.softplus(torch.tensor(float(v), dtype=torch.float64)).item()  # noqa: E731
        self.above, self.below = softplus(p), 0.5 + softplus(q)
        self.up = Linear(up, up_bias, dtype=dtype, device=device)
        self.down = Linear(_pad(down.detach(), down.shape[0], self.up.n), down_bias, dtype=dtype, device=device)

    def __call__(self, x: torch.Tensor) -> torch.Tensor:
        return self.down(ops.gemm_xielu(x, self.up.w, self.up.bias, self.above, self.below))

    def tensors(self):
        yield from self.up.tensors()
        yield from self.down.tensors()


class RoutedExperts:
    """Mixture of ``ClampedGLU`` experts: fp32 softmax router over experts and ``identity`` outputs that return the input itself; the
    ``top`` best by score + correction inside the ``keep`` best of ``groups`` groups of neighbours, weighted by their scores without
    it; a shared expert for every token.  experts: (gate, up, down) each; shared: the same and its limit, or None.  ``sigmoid``: scores are
    sigmoids of the logits; ``normalize``: the weights are the scores over the chosen ones' sum; ``weigh_input``: a weight multiplies
    its expert's input instead of the output.  limit inf, alpha 1 and offset 0 make an expert a plain silu-gated unit.

    A call returns an ``ops.Mixture``: the residual update sums it."""

    TILE_PAIRS = 16  # pairs per expert from which the experts run in tiles and the shared expert in launches of its own

    def __init__(self, experts, router, correction, *, top: int, limit: float, groups: int = 1, keep: int = 1, identity: int = 0, shared=None,
                 alpha: float = 1.702, offset: float = 1.0, sigmoid: bool = False, normalize: bool = True, weigh_input: bool = False,
                 dtype=BF16, device="cuda"):
        n, k = len(experts), router.shape[1]
        entries = (router.shape[0], n + identity if correction is None else correction.numel())
        if entries != (n + identity, n + identity):
            raise ValueError(f"router and correction have {entries[0]} and {entries[1]} entries, {n + identity} expected")
        if n < 1 or not 1 <= top <= min(n + identity, 64) or n + identity > 1024:
            raise ValueError("between 1 and 1024 outputs and a top of at most 64 of them are supported")
        if groups < 1 or (n + identity) % groups or not 1 <= keep <= groups or groups > 64:
            raise ValueError("groups (at most 64) must divide the router's outputs, and 1 to all of them be kept")
        if keep * ((n + identity) // groups) < top:
            raise ValueError("the kept groups hold fewer outputs than a token uses")
        if weigh_input and identity:
            raise ValueError("identity outputs return their input: weights on the inputs do not reach them")
        self.flags, self.weigh_input = (ROUTER_SIGMOID if sigmoid else 0) | (0 if normalize else ROUTER_PLAIN), weigh_input
        self.experts, self.top, self.groups, self.keep = n, top, groups, keep
        self.width, self.k, self.ff = experts[0][2].shape[0], ops.round8(k), ops.round8(experts[0][0].shape[0])
        self.dtype, self.device = dtype, device
        dev = lambda w, rows, cols: _pad(w.detach().to(device=device, dtype=dtype), rows, cols).contiguous()  # noqa: E731
        gates, ups, downs = ([dev(e[i], *size) for e in experts] for i, size in
                             ((0, (self.ff, self.k)), (1, (self.ff, self.k)), (2, (ops.round8(self.width), self.ff))))
        if dtype == F32:
            self.gate_up, self.down = (torch.stack(gates), torch.stack(ups)), torch.stack(downs)
        else:
            self.gate_up = torch.stack([ops.pack_gate_up(g, u).data for g, u in zip(gates, ups)])
            self.down = torch.stack([ops.pack_rows(d) for d in downs])
        self.router = dev(router, n + identity, self.k)
        self.correction = None if correction is None else correction.detach().to(device=device, dtype=F32).contiguous()
        self.glu = OharaGlu(limit, alpha, offset, 0)
        self.shared = None if shared is None else ClampedGLU(*shared[:3], limit=shared[3], alpha=alpha, offset=offset, dtype=dtype,
                                                             device=device)
        self._counter = torch.zeros(1, dtype=torch.int32, device=device)
        self.trace = None  # a list: a call appends (chosen outputs, weights)

    def __call__(self, x: torch.Tensor) -> ops.Mixture:
        rows, n8 = x.shape[0], ops.round8(self.width)
        pairs = rows * self.top
        idx, w, offs, pair_of, pos_of = ops.moe_router(x, self.router, self.correction, self.k, self.top, self.groups, self.keep,
                                                       self._counter, self.flags)
        if self.trace is not None:
            self.trace.append((idx, w))
        empty = lambda *s: torch.empty(*s, dtype=self.dtype, device=x.device)  # noqa: E731
        act, y = empty(pairs, self.ff), empty(pairs, n8)
        p, glu, shared, pair_w = ops._ptr, ctypes.byref(self.glu), None, w if self.weigh_input else None
        if self.dtype == F32:
            check(lib().ohara_moe_glu_f32(p(x), x.stride(0), p(self.gate_up[0]), p(self.gate_up[1]), self.experts, self.ff, self.k, self.top,
                                          pairs, p(offs), p(pair_of), p(pair_w), glu, p(act), self.ff, ops._stream()), "moe_glu")
            check(lib().ohara_moe_down_f32(p(act), self.ff, p(self.down), self.experts, n8, self.ff, pairs, p(offs), p(y), n8,
                                           ops._stream()), "moe_down")
            if self.shared is not None:
                shared = self.shared(x)
        else:
            up, down = (0, 0, 0, None, 0, 0), (0, 0, 0, 0, 0, 0, 0)  # the shared expert's part of the launches
            if self.shared is not None and pairs >= self.TILE_PAIRS * self.experts:
                shared = self.shared(x)
            elif self.shared is not None:
                s = self.shared
                act_s, shared = empty(rows, s.ff), empty(rows, n8)
                up = (p(s.gate_up.data), s.ff, rows, ctypes.byref(OharaGlu(*s.constants, 0)), p(act_s), s.ff)
                down = (p(s.down.w.data), s.ff, rows, p(act_s), s.ff, p(shared), n8)
            check(lib().ohara_moe_glu_bf16(p(x), x.stride(0), p(self.gate_up), self.gate_up.stride(0) * 2, self.experts, self.ff, self.k,
                                           self.top, pairs, p(offs), p(pair_of), p(pair_w), glu, p(act), self.ff, *up, ops._stream()), "moe_glu")
            check(lib().ohara_moe_down_bf16(p(act), self.ff, p(self.down), self.down.stride(0) * 2, self.experts, n8, self.ff, pairs, p(offs),
                                            p(y), n8, *down, ops._stream()), "moe_down")
        return ops.Mixture(idx, None if self.weigh_input else w, pos_of, y, x, shared, self.experts)

    def tensors(self):
        yield from (self.gate_up if self.dtype == F32 else (self.gate_up,))
        yield from (t for t in (self.down, self.router, self.correction) if t is not None)
        if self.shared is not None:
            yield from self.shared.tensors()


def added(y) -> dict:
    """What ``ops.residual_norm`` needs to add y (a tensor or an ``ops.Mixture``) as it is."""
    return {"mix" if isinstance(y, ops.Mixture) else "y": y}


class GroupNorm:
    """RMS norm in ``groups`` equal runs of the row, times w and, if given, ``scale`` (applied inside ``ops.residual_norm``)."""

    def __init__(self, w, groups: int, eps: float, device="cuda", scale=None):
        if w.numel() % groups:
            raise ValueError("norm groups must divide the width")
        self.w = w.detach().to(device=device, dtype=F32).contiguous()
        if scale is not None:
            self.w = self.w * scale.detach().to(device=device, dtype=F32)
        self.groups, self.eps = groups, float(eps)

    def of(self, y) -> dict:
        """What ``ops.residual_norm`` needs to add the norm of y (a tensor or an ``ops.Mixture``)."""
        return dict(added(y), norm_w=self.w, groups=self.groups, eps=self.eps)

    def out(self) -> dict:
        """What ``ops.residual_norm`` needs to return the norm of the residual."""
        return dict(mode="norm", norm2_w=self.w, groups=self.groups, eps=self.eps)


class LayerNorm(GroupNorm):
    """(x - mean) / sqrt(variance + eps) times w, no bias (applied inside ``ops.residual_norm``)."""

    def __init__(self, w, eps: float, device="cuda"):
        super().__init__(w, 1, eps, device)

    def of(self, y) -> dict:
        return dict(super().of(y), center_y=True)

    def out(self) -> dict:
        return dict(super().out(), center_out=True)


class InputConv:
    """h + causal depthwise convolution of h over time; w (width, taps), the last column is the current token's."""

    def __init__(self, w, device="cuda"):
        self.w = w.detach().to(device=device, dtype=F32).t().contiguous()  # (taps, width)
        self.device = device

    def state(self, rows: int) -> torch.Tensor:
        taps, width = self.w.shape
        return torch.zeros(rows, taps, width, dtype=F32, device=self.device)

    def __call__(self, x, ring, seq: ops.Seq, dtype):
        return ops.input_conv(x, self.w, ring, seq, dtype)


def distance_slopes(heads: int) -> torch.Tensor:
    """2^(-8 (h + 1) / heads) for head h: the slopes of a linear distance bias (ALiBi)."""
    return torch.tensor([2.0 ** (-8.0 * (h + 1) / heads) for h in range(heads)], dtype=F32)


class CachedAttention:
    """Keys and values per position, and the split of a decode step's context, for the attention classes below."""

    WORKGROUPS = 1024   # decode: a context is cut into chunks until about this many workgroups run
    MIN_CHUNK = 128     # positions of a chunk at least (of what a query can see of the cache's capacity)

    def _sizes(self, heads: int, kv_heads: int, dim: int, vdim: int, projections, dtype, device) -> None:
        if heads < 1 or kv_heads < 1 or heads % kv_heads:
            raise ValueError("kv_heads must divide heads")
        for name, w, n in projections:
            if w.shape[0] != n:
                raise ValueError(f"attention {name} projection has {w.shape[0]} rows, {n} expected")
        if max(dim, vdim) > 256:
            raise ValueError("attention head sizes up to 256 are supported")
        self.heads, self.kv_heads, self.dim, self.vdim = heads, kv_heads, dim, vdim
        self.dtype, self.device = dtype, device
        self._ws: dict = {}

    def _visible(self, max_seq_length: int) -> int:
        return max_seq_length

    def state(self, rows: int, max_seq_length: int) -> dict:
        zeros = lambda n: torch.zeros(rows, max_seq_length, self.kv_heads, ops.round8(n), dtype=self.dtype, device=self.device)  # noqa: E731
        self._split(rows, max_seq_length)  # a step captured before any eager one finds its workspace initialised
        return {"key": zeros(self.dim), "value": zeros(self.vdim)}

    def _head_sets(self) -> int:
        """Sets of query heads of one KV head (up to four) that a workgroup of a decode step serves."""
        rep = self.heads // self.kv_heads
        return self.kv_heads * -(-rep // (4 if rep >= 4 else (2 if rep >= 2 else 1)))

    def n_split(self, batch: int, max_seq_length: int) -> int:
        return max(1, min(64, self.WORKGROUPS // (batch * self._head_sets()), self._visible(max_seq_length) // self.MIN_CHUNK))

    def _split(self, batch: int, max_seq_length: int):
        """(chunks, workspace) of a decode step; steps of the same batch size share the workspace, so they must run on one
        stream or otherwise in turn."""
        ns = self.n_split(batch, max_seq_length)
        if ns == 1:
            return 1, None
        ws = self._ws.get((batch, ns))
        if ws is None:
            ws = self._ws[(batch, ns)] = ops.attn_bias_workspace(batch, self.heads, self.vdim, ns, self.device)
        return ns, ws


class BiasedAttention(CachedAttention):
    """Causal attention without rotation: q and k normed over the whole projection, values over each head without a
    weight, a linear distance bias on the scores, one sigmoid gate per head on the outputs.

    q, k, v, gate, out: (weight, bias or None) pairs of the projections off the same input."""

    def __init__(self, q, k, v, gate, out, q_norm, k_norm, *, heads: int, kv_heads: int, dim: int, vdim: int, scale: float,
                 eps: float, slopes: torch.Tensor, dtype=BF16, device="cuda"):
        parts = (("q", q, heads * dim), ("k", k, kv_heads * dim), ("v", v, kv_heads * vdim), ("gate", gate, heads))
        self._sizes(heads, kv_heads, dim, vdim, [(name, t, n) for name, pair, n in parts for t in pair if t is not None], dtype, device)
        self.scale, self.eps = float(scale), float(eps)
        pairs = (q, k, v, gate)
        biases = [b if b is not None else torch.zeros(w.shape[0], dtype=w.dtype, device=w.device) for w, b in pairs]
        has_bias = any(b is not None for _, b in pairs)
        self.proj = Linear(torch.cat([w for w, _ in pairs]), torch.cat(biases) if has_bias else None, dtype=dtype, device=device)
        self.out = Linear(out, dtype=dtype, device=device)
        dev = lambda t: t.detach().to(device=device, dtype=F32).contiguous()  # noqa: E731
        self.q_norm, self.k_norm, self.slopes = dev(q_norm), dev(k_norm), dev(slopes)
        self.gate_at = heads * dim + kv_heads * (dim + vdim)

    def __call__(self, h, state, seq: ops.Seq):
        p = self.proj(h)
        q = ops.qkv_norm_append(p, self.heads, self.kv_heads, self.dim, self.vdim, self.q_norm, self.k_norm, self.eps,
                                state.key, state.value, seq)
        ns, ws = self._split(seq.batch, state.key.shape[1]) if seq.seq_len == 1 else (1, None)
        gate = p[:, self.gate_at:self.gate_at + self.heads]
        att = ops.attn_bias(q, state.key, state.value, self.heads, self.kv_heads, self.dim, self.vdim, self.scale, self.slopes,
                            gate, seq, ns, ws)
        return self.out(att)

    def tensors(self):
        yield from self.proj.tensors()
        yield from self.out.tensors()
        yield from (self.q_norm, self.k_norm)


_ROTARY: dict = {}


def scaled_frequencies(f: torch.Tensor, factor: float, low: float, high: float, original: float) -> torch.Tensor:
    """Rotary frequencies stretched to longer contexts as in Llama 3.1: those that turn at least ``high`` times in ``original``
    positions stay, those that turn at most ``low`` times are divided by ``factor``, in between the two are mixed linearly."""
    turns = original * f / (2 * math.pi)
    if high <= low:
        return torch.where(turns < low, f / factor, f)
    s = ((turns - low) / (high - low)).clamp(0, 1)
    return (1 - s) * f / factor + s * f


@dataclass(frozen=True)
class Yarn:
    """Rotary frequencies for longer contexts by the index of the pair (YaRN): pairs that turn more than ``fast`` times in ``original``
    positions stay, those below ``slow`` turns are divided by ``factor``, a ramp over the indices between; cos and sin grow by
    0.1 ln(factor) + 1."""

    factor: float
    fast: float
    slow: float
    original: float

    def apply(self, f: torch.Tensor, base: float, dims: int) -> tuple[torch.Tensor, float]:
        index = lambda turns: dims * math.log(self.original / (2 * math.pi * turns)) / (2 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(index(self.fast)), 0), min(math.ceil(index(self.slow)), dims - 1)
        ramp = ((torch.arange(len(f), dtype=f.dtype) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        return f / self.factor * ramp + f * (1 - ramp), 0.1 * math.log(self.factor) + 1.0


def rotary_tables(base: float, dims: int, positions: int, device, scaling: tuple | Yarn | None = None):
    """(cos, sin) of position * base^(-2i / dims), i < dims / 2, as (positions, dims / 2) fp32; one pair for all layers that share
    the constants.  ``scaling``: (factor, low, high, original) of ``scaled_frequencies``, or a ``Yarn``."""
    device = torch.device(device)
    key = (float(base), dims, positions, device.type, device.index, scaling)
    if key not in _ROTARY:
        f = float(base) ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64) / max(dims, 1))
        magnitude = 1.0
        if isinstance(scaling, Yarn):
            f, magnitude = scaling.apply(f, float(base), dims)
        elif scaling is not None:
            f = scaled_frequencies(f, *scaling)
        a = torch.arange(positions, dtype=torch.float64).unsqueeze(1) * f
        _ROTARY[key] = tuple((magnitude * t).to(device, F32).contiguous() for t in (a.cos(), a.sin()))
    return _ROTARY[key]


def neighbours_of_halves(w: torch.Tensor, dim: int, rot_dims: int) -> torch.Tensor:
    """Rows of heads of ``dim`` whose pairs are (i, i + rot_dims / 2) -> the same with pairs (2i, 2i + 1).  Scores do not change when q and
    k are reordered alike."""
    order = torch.arange(dim)
    order[:rot_dims] = order[:rot_dims].view(2, -1).t().reshape(-1)
    return w.unflatten(0, (-1, dim))[:, order.to(w.device)].flatten(0, 1)


class RotaryAttention(CachedAttention):
    """Causal attention with the first ``rot_dims`` dimensions of q and k rotated in neighbouring pairs (``rot_halves``: i with
    i + rot_dims / 2; ``rot_scaling``: of ``rotary_tables``), soft-capped scores (``cap``, 0: none), with ``chunk`` > 0 keys of the query's own chunk of that many positions
    only, with ``window`` > 0 only that many keys up to the query's own.  q_norm, k_norm: every q / k head over its own root mean
    square times these first.  sinks: per head a score that joins the softmax without a value.  ``bare``: the projections are a
    ``ParallelMixer``'s, which scales the heads' outputs by ``out_scale``."""

    def __init__(self, q, k, v, out, *, heads: int, kv_heads: int, dim: int, vdim: int, scale: float, rot_base: float, rot_dims: int,
                 cap: float = 0.0, chunk: int = 0, window: int = 0, q_norm=None, k_norm=None, eps: float = 0.0, sinks=None,
                 rot_scaling: tuple | Yarn | None = None, rot_halves: bool = False, bare: bool = False, dtype=BF16, device="cuda"):
        self._sizes(heads, kv_heads, dim, vdim, (("q", q, heads * dim), ("k", k, kv_heads * dim), ("v", v, kv_heads * vdim)), dtype, device)
        if rot_dims < 0 or rot_dims % 2 or rot_dims > dim:
            raise ValueError("rotated dimensions must be an even number up to the head size")
        if cap < 0 or chunk < 0 or window < 0:
            raise ValueError("soft cap, chunk and window sizes cannot be negative")
        if (q_norm is None) != (k_norm is None) or any(t is not None and t.numel() != dim for t in (q_norm, k_norm)):
            raise ValueError("head norms come for q and k, with one weight per dimension of a head")
        self.scale, self.cap, self.chunk, self.rot_base, self.rot_dims = float(scale), float(cap), chunk, float(rot_base), rot_dims
        self.window, self.eps, self.out_scale = window, float(eps), 1.0
        self.rot_scaling = rot_scaling if rot_scaling is None or isinstance(rot_scaling, Yarn) else tuple(float(v) for v in rot_scaling)
        if rot_halves:
            q, k, q_norm, k_norm = (None if t is None else neighbours_of_halves(t, dim, rot_dims) for t in (q, k, q_norm, k_norm))
        dev = lambda t: None if t is None else t.detach().to(device=device, dtype=F32).contiguous()  # noqa: E731
        self.q_norm, self.k_norm, self.sinks = dev(q_norm), dev(k_norm), dev(sinks)
        self.in_weight, self.out_weight = torch.cat([q, k, v]), out
        if not bare:
            self.proj, self.out = (Linear(w, dtype=dtype, device=device) for w in (self.in_weight, out))
            del self.in_weight, self.out_weight

    def _visible(self, max_seq_length: int) -> int:
        return min([max_seq_length] + [n for n in (self.chunk, self.window) if n])

    def _tables(self, positions: int):
        return rotary_tables(self.rot_base, self.rot_dims, positions, self.device, self.rot_scaling)

    def state(self, rows: int, max_seq_length: int) -> dict:
        self._tables(max_seq_length)
        return super().state(rows, max_seq_length)

    def heads_of(self, p, state, seq: ops.Seq, out=None):
        t_max = state.key.shape[1]
        cos, sin = self._tables(t_max)
        sizes = (self.heads, self.kv_heads, self.dim, self.vdim)
        if self.q_norm is not None:
            q = ops.qkv_headnorm_rotate_append(p, *sizes, self.q_norm, self.k_norm, self.eps, cos, sin, self.rot_dims, state.key, state.value,
                                               seq)
        else:
            q = ops.qkv_rotate_append(p, *sizes, cos, sin, self.rot_dims, state.key, state.value, seq)
        ns, ws = self._split(seq.batch, t_max) if seq.seq_len == 1 else (1, None)
        return ops.attn_scored(q, state.key, state.value, *sizes, t_max, self.scale, seq, cap=self.cap, chunk=self.chunk, window=self.window,
                               sinks=self.sinks, n_split=ns, workspace=ws, out_scale=self.out_scale, out=out)

    def __call__(self, h, state, seq: ops.Seq):
        return self.out(self.heads_of(self.proj(h), state, seq))

    def tensors(self):
        if hasattr(self, "proj"):
            yield from self.proj.tensors()
            yield from self.out.tensors()
        yield from (t for t in (self.q_norm, self.k_norm, self.sinks) if t is not None)


class MixedHeadAttention(RotaryAttention):
    """``RotaryAttention`` whose softmax weights are mixed across heads before they meet the values: head h applies sum_g talk[h, g] w_g to
    the values of its own key/value head.  temp: per head a factor of the scores.  With a window, the ``keep_first`` first positions stay
    visible behind it."""

    def __init__(self, q, k, v, out, talk, *, temp=None, keep_first: int = 0, **kw):
        super().__init__(q, k, v, out, **kw)
        if talk.shape != (self.heads, self.heads) or (temp is not None and temp.numel() != self.heads):
            raise ValueError("talk is a matrix over the heads, temp has one entry per head")
        if keep_first < 0 or self.cap or self.chunk or self.sinks is not None:
            raise ValueError("mixed heads come with a window and kept positions, without caps, chunks and sinks")
        if self.heads > 256:
            raise ValueError("up to 256 mixed heads are supported")
        dev = lambda t: t.detach().to(device=self.device, dtype=F32).contiguous()  # noqa: E731
        self.talk, self.temp, self.keep_first = dev(talk), None if temp is None else dev(temp), keep_first

    def _visible(self, max_seq_length: int) -> int:
        return min(max_seq_length, self.window + self.keep_first) if self.window else max_seq_length

    def n_split(self, batch: int, max_seq_length: int) -> int:
        tiles = -(-self._visible(max_seq_length) // 64)  # the kernels work on tiles of 64 positions
        return max(1, min(64, self.WORKGROUPS // (batch * self._head_sets()), tiles))

    def _split(self, batch: int, max_seq_length: int):
        ns = self.n_split(batch, max_seq_length)
        key = (batch, ns, max_seq_length)
        if key not in self._ws:
            self._ws[key] = ops.attn_mixed_workspace(batch, 1, self.heads, self.kv_heads, self.dim, self.vdim, max_seq_length, self.window,
                                                     self.keep_first, ns, self.dtype, self.device)
        return ns, self._ws[key]

    def heads_of(self, p, state, seq: ops.Seq, out=None):
        t_max = state.key.shape[1]
        cos, sin = self._tables(t_max)
        sizes = (self.heads, self.kv_heads, self.dim, self.vdim)
        q = ops.qkv_rotate_append(p, *sizes, cos, sin, self.rot_dims, state.key, state.value, seq)
        ns, ws = self._split(seq.batch, t_max) if seq.seq_len == 1 else (1, None)
        ends = None if seq.seq_len == 1 or seq.host is None else max(s + seq.seq_len for s in seq.host[0])
        return ops.attn_mixed(q, state.key, state.value, *sizes, self.scale, self.talk, seq, temp=self.temp, window=self.window,
                              keep=self.keep_first, positions=None if ends is None else min(ends, t_max), n_split=ns, workspace=ws)

    def tensors(self):
        yield from super().tensors()
        yield from (t for t in (self.talk, self.temp) if t is not None)


class LatentAttention:
    """Causal attention without positions whose queries come from one normed latent and whose keys and values are per-head
    projections of another, the only thing cached; every output element times a sigmoid gate.

    q_down (q_rank, width), q_up (heads * dim, q_rank); kv_down (rank, width), k_up (heads * dim, rank), v_up (heads * vdim, rank);
    gate (heads * vdim, width).  Calls of ``EXPAND`` tokens and more form keys and values of all their positions once; shorter
    ones apply k_up to the query and v_up to the weighted sum of the latents."""

    EXPAND = 16
    WORKGROUPS = 256    # a context is cut into chunks until about this many workgroups run
    TILE = 64           # positions of a chunk at least

    def __init__(self, q_down, q_norm, q_up, kv_down, kv_norm, k_up, v_up, gate, out, *, heads: int, dim: int, vdim: int, scale: float,
                 eps: float, dtype=BF16, device="cuda"):
        rq, r = q_down.shape[0], kv_down.shape[0]
        for name, w, n in (("q_up", q_up, heads * dim), ("k_up", k_up, heads * dim), ("v_up", v_up, heads * vdim), ("gate", gate, heads * vdim)):
            if w.shape[0] != n:
                raise ValueError(f"latent attention {name} projection has {w.shape[0]} rows, {n} expected")
        if max(dim, vdim) > 256 or r > 512:
            raise ValueError("latent attention head sizes up to 256 and cached latents up to 512 are supported")
        self.heads, self.dim, self.vdim, self.q_rank, self.rank = heads, dim, vdim, rq, r
        self.scale, self.eps, self.dtype, self.device = float(scale), float(eps), dtype, device
        kw = dict(dtype=dtype, device=device)
        r8 = ops.round8
        self.off_c = r8(rq)
        self.off_g = self.off_c + r8(r)
        self.proj = Linear(torch.cat([_pad(q_down, self.off_c), _pad(kv_down, r8(r)), gate]), **kw)
        self.out = Linear(out, **kw)
        self.q_up = Linear(self._per_head(q_up, dim).flatten(0, 1), **kw)
        self._up_projections(k_up, v_up)
        dev = lambda t: t.detach().to(device=device, dtype=F32).contiguous()  # noqa: E731
        self.q_norm, self.kv_norm = dev(q_norm), dev(kv_norm)

    def _per_head(self, w, n):  # (heads * n, k) -> (heads, n, k), rows and columns padded to multiples of 8
        w = w.detach().view(self.heads, n, w.shape[1])
        return F.pad(w, (0, ops.round8(w.shape[2]) - w.shape[2], 0, ops.round8(n) - n))

    def _up_projections(self, k_up, v_up) -> None:
        k_heads, v_heads = self._per_head(k_up, self.dim), self._per_head(v_up, self.vdim)
        kw = dict(dtype=self.dtype, device=self.device)
        self.kv_up = Linear(torch.cat([k_heads.flatten(0, 1), v_heads.flatten(0, 1)]), **kw)
        self.k_absorb = k_heads.transpose(1, 2).to(**kw).contiguous()
        self.v_absorb = v_heads.to(**kw).contiguous()
        self._ws: dict = {}

    def _visible(self, max_seq_length: int) -> int:
        return max_seq_length

    def state(self, rows: int, max_seq_length: int) -> dict:
        self._split(rows, max_seq_length)
        return {"latent": torch.zeros(rows, max_seq_length, ops.round8(self.rank), dtype=self.dtype, device=self.device)}

    def _split(self, rows: int, max_seq_length: int):
        """(chunks, workspace) of a call over ``rows`` query tokens; calls of as many rows share the workspace."""
        ns = max(1, min(64, self.WORKGROUPS // (rows * -(-self.heads // 16)), self._visible(max_seq_length) // self.TILE))
        if ns == 1:
            return 1, None
        ws = self._ws.get((rows, ns))
        if ws is None:
            ws = self._ws[(rows, ns)] = ops.attn_latent_workspace(rows, self.heads, self.rank, ns, self.device)
        return ns, ws

    def _expanded(self, c, state, seq: ops.Seq):
        """Keys and values of all positions of every sequence (batch, longest, [heads * dim; heads * vdim]).  ``c``: the call's own
        latents where that is all of them."""
        if c is not None:
            return self.kv_up(c), seq.seq_len
        starts, counts, rows = seq.host
        ends = [s + n for s, n in zip(starts, counts)]
        kv = torch.empty(seq.batch, max(ends), self.kv_up.n, dtype=self.dtype, device=self.device)
        for b, (row, end) in enumerate(zip(rows, ends)):
            self.kv_up(state.latent[row, :end], out=kv[b, :end])
        return kv.view(-1, self.kv_up.n), max(ends)

    def __call__(self, h, state, seq: ops.Seq):
        p = self.proj(h)
        H, n = self.heads, self.heads * self.vdim
        gate = p[:, self.off_g:self.off_g + n]
        expand = seq.seq_len >= self.EXPAND and seq.host is not None
        whole = expand and not any(seq.host[0])
        cq, c = ops.latent_front(p, self.q_rank, self.off_c, self.rank, self.q_norm, self.kv_norm, self.eps, state.latent, seq, whole)
        q = self.q_up(cq)
        if expand:
            kv, length = self._expanded(c, state, seq)
            at = ops.Seq(seq.batch, seq.seq_len, int(seq.c.pos), seq.pos_dev, bool(seq.c.pos_stride), seq.lens)
            att = ops.attn_scored(q, kv, kv[:, H * ops.round8(self.dim):], H, H, self.dim, self.vdim, length, self.scale, at, gate=gate,
                                  gate_elements=True, ld_k=kv.stride(0), ld_v=kv.stride(0))
            return self.out(att)
        ns, ws = self._split(seq.rows, state.latent.shape[1])
        mixed = ops.attn_latent(ops.head_linear(q, self.k_absorb, ops.round8(self.rank)), state.latent, H, self.rank, self.scale, seq, ns, ws)
        return self.out(ops.head_linear(mixed, self.v_absorb, self.vdim, gate))

    def tensors(self):
        for lin in (self.proj, self.q_up, self.kv_up, self.out):
            yield from lin.tensors()
        yield from (self.q_norm, self.kv_norm)


class RotaryLatentAttention(LatentAttention):
    """Latent attention with positions: every query head is dim unrotated elements followed by rot_dim elements rotated in neighbouring
    pairs, which meet one rotated key part that all heads share and that is cached behind the latent.  ``window`` > 0: that many keys up
    to the query's own.

    q (heads * (dim + rot_dim), width); k_up, v_up and out as ``LatentAttention``.  kv_down (rank + rot_dim, width) and kv_norm (rank)
    are None for a layer that reads the cached rows of another one (``borrow``), of which it needs the rank."""

    def __init__(self, q, kv_down, kv_norm, k_up, v_up, out, *, heads: int, dim: int, rot_dim: int, vdim: int, rank: int, scale: float, eps: float,
                 rot_base: float, rot_scaling=None, window: int = 0, dtype=BF16, device="cuda"):
        for name, w, shape in (("q", q, (heads * (dim + rot_dim), q.shape[1])), ("kv_down", kv_down, (rank + rot_dim, q.shape[1])),
                               ("k_up", k_up, (heads * dim, rank)), ("v_up", v_up, (heads * vdim, rank))):
            if w is not None and tuple(w.shape) != shape:
                raise ValueError(f"latent attention {name} projection is {tuple(w.shape)}, {shape} expected")
        if rank > 512 or rot_dim > 128 or rot_dim < 2 or rot_dim % 2 or window < 0:
            raise ValueError("cached latents up to 512 and an even number of rotated dimensions up to 128 are supported")
        self.heads, self.dim, self.vdim, self.rank, self.rot_dim = heads, dim, vdim, rank, rot_dim
        self.scale, self.eps, self.window, self.dtype, self.device = float(scale), float(eps), window, dtype, device
        self.rot = (float(rot_base), rot_dim, rot_scaling)
        r8 = ops.round8
        self.dq, self.dr, self.row = r8(dim), r8(rot_dim), r8(rank) + r8(rot_dim)  # of a query's parts and of a cached row
        q = q.detach().view(heads, dim + rot_dim, -1)
        parts = [torch.cat([F.pad(q[:, :dim], (0, 0, 0, self.dq - dim)), F.pad(q[:, dim:], (0, 0, 0, self.dr - rot_dim))], 1).flatten(0, 1)]
        self.n_q = heads * (self.dq + self.dr)
        if kv_down is not None:
            parts += [_pad(kv_down[:rank], r8(rank)), _pad(kv_down[rank:], self.dr)]
        self.proj = Linear(torch.cat(parts), dtype=dtype, device=device)
        self.out = Linear(out, dtype=dtype, device=device)
        self._up_projections(k_up, v_up)
        self.kv_norm = None if kv_norm is None else kv_norm.detach().to(device=device, dtype=F32).contiguous()

    def _visible(self, max_seq_length: int) -> int:
        return min(max_seq_length, self.window) if self.window else max_seq_length

    def _tables(self, positions: int):
        base, dims, scaling = self.rot
        return rotary_tables(base, dims, positions, self.device, scaling)

    def state(self, rows: int, max_seq_length: int) -> dict:
        return self.borrow({"latent": torch.zeros(rows, max_seq_length, self.row, dtype=self.dtype, device=self.device)}, rows, max_seq_length)

    def borrow(self, tensors: dict, rows: int, max_seq_length: int) -> dict:
        """The state of a layer that reads another one's."""
        if tensors["latent"].shape[2] != self.row:
            raise ValueError("the cached rows of the other layer have another size")
        self._split(rows, max_seq_length)
        self._tables(max_seq_length)
        return tensors

    def _expanded(self, rows, state, seq: ops.Seq):
        """(keys and values of all visible positions, rotated key parts, positions per sequence, the call's place among them).  ``rows``: the
        call's own cached rows where those are all positions."""
        n, r = self.kv_up.n, ops.round8(self.rank)
        if rows is not None:
            return self.kv_up(rows[:, :r]), rows[:, r:], seq.seq_len, ops.Seq(seq.batch, seq.seq_len, lens=seq.lens)
        starts, counts, slots = seq.host
        firsts = [max(0, s - self.window + 1) if self.window else 0 for s in starts]
        length = max(s - f for s, f in zip(starts, firsts)) + seq.seq_len
        kv = torch.empty(seq.batch, length, n + self.dr, dtype=self.dtype, device=self.device)
        for b, (slot, s, f, count) in enumerate(zip(slots, starts, firsts, counts)):
            cached, own = state.latent[slot, f:s + count], kv[b, :s - f + count]
            self.kv_up(cached[:, :r], out=own[:, :n])
            own[:, n:] = cached[:, r:]
        kv = kv.view(-1, n + self.dr)
        at = torch.tensor([s - f for s, f in zip(starts, firsts)], dtype=torch.int32).to(kv.device)
        return kv, kv[:, n:], length, ops.Seq(seq.batch, seq.seq_len, 0, at, True, seq.lens)

    def __call__(self, h, state, seq: ops.Seq):
        p = self.proj(h)
        H, dq, dr, r, cache = self.heads, self.dq, self.dr, ops.round8(self.rank), state.latent
        cos, sin = self._tables(cache.shape[1])
        expand = seq.seq_len >= self.EXPAND and seq.host is not None and max(dq + dr, self.vdim) <= 256
        whole = expand and not any(seq.host[0])
        # the rotated parts of the queries stay in their place, or go behind the queries on the latents
        q = p[:, :self.n_q] if expand else torch.empty(p.shape[0], H * self.row, dtype=p.dtype, device=p.device)
        at, stride = (q[:, dq:], dq + dr) if expand else (q[:, r:], self.row)
        own = {} if self.kv_norm is None else dict(cache=cache, off_c=self.n_q, off_r=self.n_q + r, rank=self.rank, cn=self.kv_norm, eps=self.eps,
                                                   compact=whole)
        rows = ops.latent_rotary_front(p, H, dq, cos, sin, at, stride, seq, **own)
        if expand:
            if rows is not None:
                seq.carry[cache.data_ptr()] = rows
            kv, part, length, place = self._expanded(seq.carry.get(cache.data_ptr()) if whole else None, state, seq)
            return self.out(ops.attn_scored(q, kv, kv[:, H * dq:], H, H, dq + dr, self.vdim, length, self.scale, place, window=self.window,
                                            ld_k=kv.stride(0), ld_v=kv.stride(0), k_shared=part, ld_shared=part.stride(0), d_shared=dr))
        ops.head_linear(p, self.k_absorb, r, out=q, x_heads=dq + dr, out_heads=self.row)
        ns, ws = self._split(seq.rows, cache.shape[1])
        mixed = ops.attn_latent(q, cache, H, self.rank, self.scale, seq, ns, ws, window=self.window)
        return self.out(ops.head_linear(mixed, self.v_absorb, self.vdim))

    def tensors(self):
        for lin in (self.proj, self.kv_up, self.out):
            yield from lin.tensors()
        if self.kv_norm is not None:
            yield self.kv_norm


class TokenSide:
    """What a layer adds to the residual for its token: proj(gelu_tanh(gate x) * e) with e the row's ``dim`` entries of an embedding
    table from ``column`` on, over its own root mean square times norm_w (``norm``)."""

    ONE_CU = 1 << 16  # elements of either matrix up to which a single workgroup reads them as fast as several launches do

    def __init__(self, gate, proj, norm_w, table, column: int, *, eps: float, dtype=BF16, device="cuda"):
        self.gate, self.proj = Linear(gate, dtype=dtype, device=device), Linear(proj, dtype=dtype, device=device)
        self.norm = GroupNorm(norm_w, 1, eps, device)
        self.table, self.column = table, column

    @staticmethod
    def lay_out(table, layers: int, *, dtype=BF16, device="cuda") -> torch.Tensor:
        """(vocab, layers * dim) -> (vocab, layers * dim rounded up to 8), each layer's entries followed by zeros."""
        vocab, n = table.shape
        t = table.detach().view(vocab, layers, n // layers)
        return F.pad(t, (0, ops.round8(t.shape[2]) - t.shape[2])).flatten(1).to(device=device, dtype=dtype).contiguous()

    def __call__(self, x, ids):
        return self.proj(ops.gemm_gelu_lookup(x, self.gate.w, self.table, self.column, ids))

    def update(self, x, seq: ops.Seq, ids, y, norm, after):
        """The residual x plus norm(y), plus what the side embedding makes of that; returns ``after`` of it (``norm``, ``after``:
        norms over the whole row with this one's eps).  One launch where the sizes allow it; a few rows of a wide model take
        four, whose weights more than one CU reads."""
        rows, d = x.shape
        same = norm.groups == after.groups == 1 and norm.eps == after.eps == self.norm.eps
        fits = d % 4 == 0 and d <= ops.TOKEN_SIDE_ELEMENTS and self.gate.n <= 256
        if self.gate.dtype == BF16 and same and fits and (rows > 64 or self.gate.n * d <= self.ONE_CU):
            return ops.token_side(x, y, norm.w, self.gate.w, self.proj.w, self.table, self.column, ids, self.norm.w, norm.eps, after.w,
                                  center_y=isinstance(norm, LayerNorm), center_out=isinstance(after, LayerNorm))
        h = ops.residual_norm(x, seq, self.gate.dtype, **{**norm.of(y), "mode": "copy"})
        return ops.residual_norm(x, seq, self.gate.dtype, **{**self.norm.of(self(h, ids)), **after.out()})

    def tensors(self):
        yield from self.gate.tensors()
        yield from self.proj.tensors()
        yield self.norm.w


class DeltaRule:
    """Gated delta rule (see csrc/delta_rule.hip for the equations): short convolutions with silu on q, k and v, unit q and k,
    gated norm per head.  The subclasses give decays and output gates."""

    WORKSPACE = 1 << 30  # bytes of per-chunk intermediates at most; longer prompts are walked in segments
    _workspaces: dict = {}  # device -> the workspace every layer on that device shares (prompts run on one stream)

    def _sizes(self, heads: int, kv_heads: int, dim: int, vdim: int, q, k, v, more, convs, a_log, dt_bias, norm_w, eps: float, dtype, device):
        if heads < 1 or kv_heads < 1 or heads % kv_heads:
            raise ValueError("kv_heads must divide heads")
        for name, w, n in (("q", q, kv_heads * dim), ("k", k, kv_heads * dim), ("v", v, heads * vdim), *more):
            if w.shape[0] != n:
                raise ValueError(f"delta rule {name} projection has {w.shape[0]} rows, {n} expected")
        if max(dim, vdim) > 256:
            raise ValueError("delta rule head sizes up to 256 are supported")
        self.heads, self.kv_heads, self.dim, self.vdim = heads, kv_heads, dim, vdim
        self.dtype, self.device = dtype, torch.device(device)
        self.channels = 2 * kv_heads * dim + heads * vdim
        self.taps = convs[0].shape[1]
        self.off_a = ops.round8(self.channels)
        self.conv_w = self._dev(torch.cat(convs).t())
        self.neg_a = -torch.exp(self._dev(a_log))
        self.dt_bias, self.norm_w = self._dev(dt_bias), self._dev(norm_w)
        d = OharaDelta()
        d.heads, d.kv_heads, d.dim, d.vdim, d.taps, d.eps = heads, kv_heads, dim, vdim, self.taps, float(eps)
        d.conv_w, d.neg_a, d.dt_bias, d.norm_w = (t.data_ptr() for t in (self.conv_w, self.neg_a, self.dt_bias, self.norm_w))
        self._c = d

    def _dev(self, t, dtype=F32):
        return t.detach().to(device=self.device, dtype=dtype).contiguous()

    def state(self, rows: int, max_seq_length: int) -> dict:
        return {"delta": torch.zeros(rows, self.heads, self.dim, (self.vdim + 3) // 4 * 4, dtype=F32, device=self.device),
                "ring": torch.zeros(rows, self.taps, self.channels, dtype=self.dtype, device=self.device)}

    def _workspace(self, batch: int, tokens: int) -> torch.Tensor:
        need = ops.delta_workspace_bytes(self.heads, self.dim, self.vdim, batch, tokens)
        need = max(min(need, self.WORKSPACE), ops.delta_workspace_bytes(self.heads, self.dim, self.vdim, batch, 1))
        ws = DeltaRule._workspaces.get(self.device)
        if ws is None or ws.numel() < need:
            ws = DeltaRule._workspaces[self.device] = torch.empty(need, dtype=torch.uint8, device=self.device)
        return ws

    def _low_rank(self, p):
        """(decay logits, output gates) of a prompt that are not columns of p."""
        return None, None

    def __call__(self, h, state, seq: ops.Seq):
        p = self.proj(h)
        if seq.seq_len == 1:
            return self.out(ops.delta_step(self._c, p, state.delta, state.ring, seq))
        za, zg = self._low_rank(p)
        o = ops.delta_prefill(self._c, p, za, zg, state.delta, state.ring, self._workspace(seq.batch, seq.seq_len), seq)
        return self.out(o)

    def tensors(self):
        yield from self.proj.tensors()
        yield from self.out.tensors()
        yield from (self.conv_w, self.neg_a, self.dt_bias, self.norm_w)


class ChannelDelta(DeltaRule):
    """One decay per head and key channel, low-rank decay and output-gate projections, sigmoid gate.  q, k: (kv_heads * dim, width);
    v: (heads * vdim, width); convs: (channels, taps) each."""

    def __init__(self, q, k, v, q_conv, k_conv, v_conv, beta, a_log, a1, a2, dt_bias, g1, g2, norm_w, out, *, heads: int,
                 kv_heads: int, dim: int, vdim: int, eps: float, dtype=BF16, device="cuda"):
        self._sizes(heads, kv_heads, dim, vdim, q, k, v, (("beta", beta, heads), ("a2", a2, heads * dim), ("g2", g2, heads * vdim)),
                    (q_conv, k_conv, v_conv), a_log, dt_bias, norm_w, eps, dtype, device)
        ra, rg = ops.round8(a1.shape[0]), ops.round8(g1.shape[0])
        self.off_g, self.off_b = self.off_a + ra, self.off_a + ra + rg
        qkv = _pad(torch.cat([q, k, v]), self.off_a)
        self.proj = Linear(torch.cat([qkv, _pad(a1, ra), _pad(g1, rg), beta]), dtype=dtype, device=device)
        a2, g2 = _pad(a2, a2.shape[0], ra), _pad(g2, g2.shape[0], rg)
        self.a2_proj, self.g2_proj = (Linear(w, dtype=dtype, device=device) for w in (a2, g2))
        self.out = Linear(out, dtype=dtype, device=device)
        self.a2, self.g2 = self._dev(a2, dtype), self._dev(g2, dtype)
        d = self._c
        d.rank_a, d.rank_g, d.off_a, d.off_g, d.off_b = ra, rg, self.off_a, self.off_g, self.off_b
        d.a2, d.g2 = self.a2.data_ptr(), self.g2.data_ptr()

    def _low_rank(self, p):
        return self.a2_proj(p[:, self.off_a:self.off_g]), self.g2_proj(p[:, self.off_g:self.off_b])

    def tensors(self):
        yield from super().tensors()
        for lin in (self.a2_proj, self.g2_proj):
            yield from lin.tensors()


class HeadDelta(DeltaRule):
    """One decay per head, output gate by a projection of its own through silu.  q, k: (kv_heads * dim, width); v, gate:
    (heads * vdim, width); beta, decay: (heads, width); convs: (channels, taps) each."""

    def __init__(self, q, k, v, q_conv, k_conv, v_conv, beta, a_log, decay, dt_bias, gate, norm_w, out, *, heads: int, kv_heads: int,
                 dim: int, vdim: int, eps: float, dtype=BF16, device="cuda"):
        self._sizes(heads, kv_heads, dim, vdim, q, k, v, (("beta", beta, heads), ("decay", decay, heads), ("gate", gate, heads * vdim)),
                    (q_conv, k_conv, v_conv), a_log, dt_bias, norm_w, eps, dtype, device)
        self.proj = Linear(torch.cat([_pad(torch.cat([q, k, v]), self.off_a), gate, decay, beta]), dtype=dtype, device=device)
        self.out = Linear(out, dtype=dtype, device=device)
        d, n = self._c, heads * vdim
        d.off_g, d.off_a, d.off_b = self.off_a, self.off_a + n, self.off_a + n + heads
        d.flags = DELTA_SILU_GATE


class Retention:
    """Linear attention with one fixed decay per head (see csrc/retention.hip): S <- decay S + k_scale k v^T, o = S^T q, every head's o
    over its own root mean square, times silu of the gate.  q, k: (heads * dim, width); v, gate: (heads * vdim, width); out: (width,
    heads * vdim).  ``bare``: as ``RotaryAttention``."""

    WORKSPACE = 1 << 30  # bytes of chunk states at most; longer prompts are worked on in segments
    _workspaces: dict = {}  # device -> the workspace every layer on that device shares (prompts run on one stream)

    def __init__(self, q, k, v, gate, out, *, heads: int, dim: int, vdim: int, decay, k_scale: float, eps: float, bare: bool = False,
                 dtype=BF16, device="cuda"):
        for name, w, n in (("q", q, heads * dim), ("k", k, heads * dim), ("v", v, heads * vdim), ("gate", gate, heads * vdim)):
            if w.shape[0] != n:
                raise ValueError(f"retention {name} projection has {w.shape[0]} rows, {n} expected")
        if out.shape[1] != heads * vdim:
            raise ValueError(f"retention output projection has {out.shape[1]} columns, {heads * vdim} expected")
        if max(dim, vdim) > 256:
            raise ValueError("retention head sizes up to 256 are supported")
        decay = torch.as_tensor(decay, dtype=torch.float64).reshape(-1)
        if decay.numel() != heads or not bool(((decay >= 0) & (decay <= 1)).all()):
            raise ValueError("one decay between 0 and 1 per head is required")
        self.heads, self.dim, self.vdim = heads, ops.round8(dim), ops.round8(vdim)
        self.dtype, self.device = dtype, torch.device(device)

        def per_head(w, n):  # (heads * n, width) -> heads of round8(n) rows
            return F.pad(w.detach().view(heads, n, -1), (0, 0, 0, ops.round8(n) - n)).flatten(0, 1)

        self.in_weight = torch.cat([per_head(w, n) for w, n in ((q, dim), (k, dim), (v, vdim), (gate, vdim))])
        self.out_weight = F.pad(out.detach().view(-1, heads, vdim), (0, self.vdim - vdim)).flatten(1)
        self.powers = (decay.unsqueeze(1) ** torch.arange(RETENTION_CHUNK + 1, dtype=torch.float64)).to(self.device, F32).contiguous()
        nk, nv = heads * self.dim, heads * self.vdim
        self._c = OharaRetention(heads, self.dim, self.vdim, vdim, 0, nk, 2 * nk, 2 * nk + nv, eps, k_scale, 1.0, 0, self.powers.data_ptr())
        if not bare:
            self.proj, self.out = (Linear(w, dtype=dtype, device=device) for w in (self.in_weight, self.out_weight))
            del self.in_weight, self.out_weight

    @property
    def out_scale(self) -> float:
        return self._c.out_scale

    @out_scale.setter
    def out_scale(self, value: float) -> None:
        self._c.out_scale = value

    def state(self, rows: int, max_seq_length: int) -> dict:
        return {"retention": torch.zeros(rows, self.heads, self.dim, self.vdim, dtype=F32, device=self.device)}

    def _workspace(self, batch: int, tokens: int) -> torch.Tensor:
        size = lambda n: ops.retention_workspace_bytes(self.heads, self.dim, self.vdim, batch, n)  # noqa: E731
        need = max(min(size(tokens), self.WORKSPACE), size(1))
        ws = Retention._workspaces.get(self.device)
        if ws is None or ws.numel() < need:
            ws = Retention._workspaces[self.device] = torch.empty(need, dtype=torch.uint8, device=self.device)
        return ws

    def heads_of(self, p, state, seq: ops.Seq, out=None):
        ws = None if seq.seq_len == 1 else self._workspace(seq.batch, seq.seq_len)
        return ops.retention(self._c, p, state.retention, ws, seq, out)

    def __call__(self, h, state, seq: ops.Seq):
        return self.out(self.heads_of(self.proj(h), state, seq))

    def tensors(self):
        if hasattr(self, "proj"):
            yield from self.proj.tensors()
            yield from self.out.tensors()
        yield self.powers


class _Part:
    """The tensors of a layer's state whose names start with a prefix, under the rest of their names."""

    def __init__(self, state, prefix: str):
        self._state, self._prefix = state, prefix

    def __getattr__(self, name):
        return getattr(self._state, self._prefix + name)


class ParallelMixer:
    """left_scale * left(h) + right_scale * right(h) for two mixers built ``bare``: their input projections are one product, and so are
    their output projections (the scales are applied to the heads, before those are rounded)."""

    def __init__(self, left, right, left_scale: float, right_scale: float, *, dtype=BF16, device="cuda"):
        self.parts = (("left_", left), ("right_", right))
        left.out_scale, right.out_scale = float(left_scale), float(right_scale)
        r8 = ops.round8
        self.n_in, self.n_out = r8(left.in_weight.shape[0]), r8(left.out_weight.shape[1])
        self.width_out = self.n_out + r8(right.out_weight.shape[1])
        pad_cols = lambda w: _pad(w, w.shape[0], r8(w.shape[1]))  # noqa: E731
        self.proj = Linear(torch.cat([_pad(left.in_weight, self.n_in), right.in_weight]), dtype=dtype, device=device)
        self.out = Linear(torch.cat([pad_cols(left.out_weight), pad_cols(right.out_weight)], 1), dtype=dtype, device=device)
        for _, part in self.parts:
            del part.in_weight, part.out_weight

    def state(self, rows: int, max_seq_length: int) -> dict:
        return {prefix + name: t for prefix, part in self.parts for name, t in part.state(rows, max_seq_length).items()}

    def __call__(self, h, state, seq: ops.Seq):
        p = self.proj(h)
        o = torch.empty(p.shape[0], self.width_out, dtype=p.dtype, device=p.device)
        for (prefix, part), src, dst in zip(self.parts, (p[:, :self.n_in], p[:, self.n_in:]), (o[:, :self.n_out], o[:, self.n_out:])):
            part.heads_of(src, _Part(state, prefix), seq, dst)
        return self.out(o)

    def tensors(self):
        for part in (self.proj, self.out, *(part for _, part in self.parts)):
            yield from part.tensors()
