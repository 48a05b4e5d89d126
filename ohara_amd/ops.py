"""Tensor-level wrappers over the C ABI (one Python function per entry point).

PyTorch is used for device memory and the current stream only; every function here
hands raw pointers to libohara_decode.so.
"""

from __future__ import annotations

import ctypes as C

import torch

from . import _lib
from ._lib import check, lib

BF16 = torch.bfloat16


def current_stream() -> int:
    """The current device's current stream as its handle.  (``torch.cuda.current_stream().cuda_stream`` makes two objects for it: 2.7 us of the host's time
    a call, where sampling a token is 13 in all and a launch's own 3; this is 0.2.)"""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


_stream = current_stream


def _ptr(t):
    return 0 if t is None else t.data_ptr()


def _need(t: torch.Tensor, dtype, name: str):
    if not t.is_cuda:
        raise ValueError(f"{name} must be a device tensor")
    if t.dtype != dtype:
        raise ValueError(f"{name} must be {dtype}, got {t.dtype}")
    if not t.is_contiguous():
        raise ValueError(f"{name} must be contiguous")


class PackedLinear:
    """A Linear weight (N, K) in the kernels' strip/kstep/lane tile order."""

    __slots__ = ("data", "n", "k", "kind")

    def __init__(self, data, n, k, kind="rows"):
        self.data, self.n, self.k, self.kind = data, n, k, kind


def pack_rows(w: torch.Tensor, perm: torch.Tensor | None = None, n_padded: int | None = None) -> torch.Tensor:
    """Pack a (N, K) bf16 matrix; ``perm`` (int32, device) maps packed row -> source row."""
    _need(w, BF16, "w")
    n, k = w.shape
    if n_padded is None:
        n_padded = (n + 15) // 16 * 16
    nbytes = C.c_int64(0)
    check(lib().ohara_pack_rows_bf16(0, n, k, k, 0, n_padded, 0, C.byref(nbytes), 0), "pack size")
    dst = torch.empty(nbytes.value // 2, dtype=BF16, device=w.device)
    check(lib().ohara_pack_rows_bf16(_ptr(w), n, k, k, _ptr(perm), n_padded, _ptr(dst), None, _stream()), "pack")
    return dst


def pack_linear(w: torch.Tensor) -> PackedLinear:
    return PackedLinear(pack_rows(w), w.shape[0], w.shape[1])


def swiglu_perm(f: int, device) -> torch.Tensor:
    fp = (f + 7) // 8 * 8
    buf = (C.c_int32 * (2 * fp))()
    check(lib().ohara_swiglu_perm(f, buf), "swiglu_perm")
    return torch.tensor(list(buf), dtype=torch.int32, device=device)


def pack_gate_up(w_gate: torch.Tensor, w_up: torch.Tensor) -> PackedLinear:
    """Interleave gate/up rows so the SwiGLU epilogue finds a gate/up pair in one lane."""
    f, k = w_gate.shape
    cat = torch.cat([w_gate, w_up], dim=0).contiguous()
    perm = swiglu_perm(f, w_gate.device)
    return PackedLinear(pack_rows(cat, perm, perm.numel()), f, k, kind="swiglu")


def pack_qkv(wq, wk, wv) -> PackedLinear:
    cat = torch.cat([wq, wk, wv], dim=0).contiguous()
    return PackedLinear(pack_rows(cat), cat.shape[0], cat.shape[1], kind="qkv")


def embed(ids: torch.Tensor, table: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    _need(table, BF16, "table")
    ids = ids.reshape(-1).contiguous()
    n, d = ids.numel(), table.shape[1]
    if out is None:
        out = torch.empty(n, d, dtype=BF16, device=table.device)
    check(lib().ohara_embed_bf16(_ptr(ids), _ptr(table), _ptr(out), n, d, table.shape[0], _stream()), "embed")
    return out


def rmsnorm(x: torch.Tensor, w: torch.Tensor, eps: float = 1e-5, out=None) -> torch.Tensor:
    _need(x, BF16, "x")
    d = x.shape[-1]
    rows = x.numel() // d
    if out is None:
        out = torch.empty_like(x)
    check(lib().ohara_rmsnorm_bf16(_ptr(x), _ptr(w), _ptr(out), rows, d, eps, _stream()), "rmsnorm")
    return out


def norm_rows(k: int) -> int:
    """Up to so many rows of this width every projection norms them itself; more may be normed ahead (ohara_projection_norm_ahead)."""
    return 64 if k <= 1024 else 32 if k <= 2048 else 16


def _normed(x, norm_w, eps, w: PackedLinear):
    """(rows, norm weight) for a projection: many rows are normed here."""
    if norm_w is not None and x.shape[0] > norm_rows(x.shape[1]):
        packed_rows = 2 * ((w.n + 7) // 8 * 8) if w.kind == "swiglu" else (w.n + 15) // 16 * 16
        if lib().ohara_projection_norm_ahead(x.shape[0], x.shape[1], packed_rows):
            return rmsnorm(x, norm_w, eps), None
    return x, norm_w


def gemm_skinny(x, w: PackedLinear, norm_w=None, eps=1e-5, residual=None, out=None) -> torch.Tensor:
    """y = [rmsnorm(x)] @ W^T (+ residual / SwiGLU epilogue by the packing kind). x: (B, K)."""
    _need(x, BF16, "x")
    x, norm_w = _normed(x, norm_w, eps, w)
    b, k = x.shape
    if k != w.k:
        raise ValueError(f"x has {k} columns, weight expects {w.k}")
    if out is None:
        out = torch.empty(b, w.n, dtype=BF16, device=x.device)
    if w.kind == "swiglu":
        epi = _lib.EPI_SWIGLU
    elif residual is not None:
        epi = _lib.EPI_RESIDUAL
    else:
        epi = _lib.EPI_STORE
    check(
        lib().ohara_gemm_skinny_bf16(
            _ptr(x), x.stride(0), _ptr(w.data), w.n, w.k, _ptr(norm_w), eps, b, epi,
            _ptr(residual), 0 if residual is None else residual.stride(0), _ptr(out), out.stride(0), _stream(),
        ),
        "gemm_skinny",
    )
    return out


def gemm(x, w: PackedLinear, residual=None, out=None) -> torch.Tensor:
    """y = x @ W^T (+ residual / SwiGLU epilogue by the packing kind) on the tiled MFMA kernel,
    for any number of rows.  x: (rows, K), rows may be strided (a column slice of a wider buffer)."""
    if not x.is_cuda or x.dtype != BF16 or x.ndim != 2 or x.stride(1) != 1:
        raise ValueError("x must be a 2-D bfloat16 device tensor with unit column stride")
    rows, k = x.shape
    if k != w.k:
        raise ValueError(f"x has {k} columns, weight expects {w.k}")
    if out is None:
        out = torch.empty(rows, w.n, dtype=BF16, device=x.device)
    epi = _lib.EPI_SWIGLU if w.kind == "swiglu" else (_lib.EPI_RESIDUAL if residual is not None else _lib.EPI_STORE)
    check(
        lib().ohara_gemm_bf16(
            _ptr(x), x.stride(0), _ptr(w.data), w.n, w.k, rows, epi,
            _ptr(residual), 0 if residual is None else residual.stride(0), _ptr(out), out.stride(0), _stream(),
        ),
        "gemm",
    )
    return out


def qkv_rope_append(x, wqkv: PackedLinear, norm_w, eps, h, h_kv, dh, cos, sin, pos, kcache, vcache,
                    q_out=None, pos_dev=None, seq_len=1, seq_pos=None):
    """x: (batch*seq_len, K) rows ordered (sequence, position).  ``seq_pos`` (int32, one entry per
    sequence, on the device) gives every sequence its own cache position instead of ``pos``."""
    _need(x, BF16, "x")
    x, norm_w = _normed(x, norm_w, eps, wqkv)
    rows = x.shape[0]
    b = rows // seq_len
    if q_out is None:
        q_out = torch.empty(rows, h * dh, dtype=BF16, device=x.device)
    t_max = kcache.shape[1]
    if seq_pos is not None:
        _need(seq_pos, torch.int32, "seq_pos")
        check(
            lib().ohara_qkv_rope_append_ragged_bf16(
                _ptr(x), x.stride(0), _ptr(wqkv.data), wqkv.k, _ptr(norm_w), eps, b, seq_len, h, h_kv, dh, _ptr(cos),
                _ptr(sin), _ptr(seq_pos), _ptr(q_out), _ptr(kcache), _ptr(vcache), t_max, _stream(),
            ),
            "qkv_rope_append_ragged",
        )
        return q_out
    check(
        lib().ohara_qkv_rope_append_bf16(
            _ptr(x), x.stride(0), _ptr(wqkv.data), wqkv.k, _ptr(norm_w), eps, b, seq_len, h, h_kv, dh, _ptr(cos), _ptr(sin),
            int(pos), _ptr(pos_dev), _ptr(q_out), _ptr(kcache), _ptr(vcache), t_max, _stream(),
        ),
        "qkv_rope_append",
    )
    return q_out


def qkv_rope(x, wqkv: PackedLinear, norm_w, eps, h, h_kv, dh, cos, sin, pos, t_max, pos_dev=None, seq_len=1):
    """As ``qkv_rope_append`` with the rotated keys and the values returned as (rows, h_kv*dh) row
    buffers instead of written into a cache -> (q, k, v)."""
    _need(x, BF16, "x")
    x, norm_w = _normed(x, norm_w, eps, wqkv)
    rows = x.shape[0]
    q = torch.empty(rows, h * dh, dtype=BF16, device=x.device)
    k = torch.empty(rows, h_kv * dh, dtype=BF16, device=x.device)
    v = torch.empty(rows, h_kv * dh, dtype=BF16, device=x.device)
    check(
        lib().ohara_qkv_rope_bf16(
            _ptr(x), x.stride(0), _ptr(wqkv.data), wqkv.k, _ptr(norm_w), eps, rows // seq_len, seq_len, h, h_kv, dh,
            _ptr(cos), _ptr(sin), int(pos), _ptr(pos_dev), t_max, _ptr(q), _ptr(k), _ptr(v), _stream(),
        ),
        "qkv_rope",
    )
    return q, k, v


def attn_workspace(batch, h, h_kv, dh, n_split, device, zeros: bool = True) -> torch.Tensor:
    n = lib().ohara_attn_workspace_bytes(batch, h, h_kv, dh, n_split)
    if n < 0:
        raise ValueError("bad attention workspace shape")
    return (torch.zeros if zeros else torch.empty)(n, dtype=torch.uint8, device=device)


def attn_cached(q, kcache, vcache, h, h_kv, dh, pos, n_split, workspace, out=None, pos_dev=None, seq_len=1,
                seq_pos=None):
    """q: (batch*seq_len, h*dh); query s of a sequence sits at cache position pos + s (or at
    seq_pos[sequence] + s when the int32 device tensor ``seq_pos`` is given)."""
    rows = q.shape[0]
    if out is None:
        out = torch.empty(rows, h * dh, dtype=BF16, device=q.device)
    if seq_pos is not None:
        _need(seq_pos, torch.int32, "seq_pos")
        check(
            lib().ohara_attn_cached_ragged_bf16(
                _ptr(q), _ptr(kcache), _ptr(vcache), rows // seq_len, seq_len, h, h_kv, dh, kcache.shape[1],
                _ptr(seq_pos), n_split, _ptr(workspace), _ptr(out), _stream(),
            ),
            "attn_cached_ragged",
        )
        return out
    check(
        lib().ohara_attn_cached_bf16(
            _ptr(q), _ptr(kcache), _ptr(vcache), rows // seq_len, seq_len, h, h_kv, dh, kcache.shape[1], int(pos),
            _ptr(pos_dev), n_split, _ptr(workspace), _ptr(out), _stream(),
        ),
        "attn_cached",
    )
    return out


def attn_prefill(q, kcache, vcache, h, h_kv, dh, pos, seq_len, out=None):
    """q: (batch*seq_len, h*dh); causal attention of seq_len queries per sequence over cache
    positions [0, pos + s] on the MFMA prefill kernels."""
    _need(q, BF16, "q")
    rows = q.shape[0]
    if out is None:
        out = torch.empty(rows, h * dh, dtype=BF16, device=q.device)
    room = max(0, lib().ohara_attn_prefill_ws_bytes(rows // seq_len, seq_len, h, h_kv, dh, int(pos)))  # < 0: refused below
    workspace = torch.empty(room, dtype=torch.uint8, device=q.device) if room else None
    check(
        lib().ohara_attn_prefill_ws_bf16(
            _ptr(q), _ptr(kcache), _ptr(vcache), rows // seq_len, seq_len, h, h_kv, dh, kcache.shape[1],
            int(pos), _ptr(out), _ptr(workspace), room, _stream(),
        ),
        "attn_prefill",
    )
    return out


def attn_auto(q, kcache, vcache, h, h_kv, dh, pos, n_split, workspace, seq_len, out=None):
    """The MFMA prefill kernels where they win, which is for many positions per sequence, else the decode kernel."""
    if lib().ohara_attn_prefill_wins(q.shape[0] // seq_len, seq_len, h, h_kv, dh, int(pos)):
        return attn_prefill(q, kcache, vcache, h, h_kv, dh, pos, seq_len, out)
    return attn_cached(q, kcache, vcache, h, h_kv, dh, pos, n_split if seq_len == 1 else 1, workspace, out, None, seq_len)


def kv_quant_append(keys, values, cache, pos, pos_dev=None, seq_pos=None):
    """keys / values (B, S, Hkv, D) bf16 -> quantised into an int8 ``KVCache`` at positions pos + s
    (``seq_pos``: one position per sequence, an int32 device tensor)."""
    _need(keys, BF16, "keys")
    _need(values, BF16, "values")
    b, s_len, hkv, d = keys.shape
    if seq_pos is not None:
        _need(seq_pos, torch.int32, "seq_pos")
        check(lib().ohara_kv_quant_append_ragged_int8(
            _ptr(keys), _ptr(values), b, s_len, hkv, d, _ptr(seq_pos), _ptr(cache.key), _ptr(cache.value), _ptr(cache.stats),
            cache.key.shape[1], _stream()), "kv_quant_append_ragged")
        return
    check(lib().ohara_kv_quant_append_int8(
        _ptr(keys), _ptr(values), b, s_len, hkv, d, int(pos), _ptr(pos_dev), _ptr(cache.key), _ptr(cache.value),
        _ptr(cache.stats), cache.key.shape[1], _stream()), "kv_quant_append")


def kv_dequant(cache, which: str, batch: int, length: int, out=None) -> torch.Tensor:
    """The first `length` positions of the int8 cache's key or value tensor as bf16 (B, length, Hkv, D)."""
    q = cache.key if which == "key" else cache.value
    _, t_max, hkv, d = q.shape
    if out is None:
        out = torch.empty(batch, length, hkv, d, dtype=BF16, device=q.device)
    check(lib().ohara_kv_dequant_int8(_ptr(q), _ptr(cache.stats), 0 if which == "key" else 1, batch, length, hkv, d, t_max,
                                      _ptr(out), _stream()), "kv_dequant")
    return out


def attn_cached_int8(q, cache, h, h_kv, dh, pos, n_split, workspace, out=None, pos_dev=None, seq_len=1, seq_pos=None):
    """attn_cached over an int8 ``KVCache`` (``seq_pos``: one position per sequence, an int32 device tensor)."""
    rows = q.shape[0]
    if out is None:
        out = torch.empty(rows, h * dh, dtype=BF16, device=q.device)
    if seq_pos is not None:
        _need(seq_pos, torch.int32, "seq_pos")
        check(lib().ohara_attn_cached_ragged_int8(
            _ptr(q), _ptr(cache.key), _ptr(cache.value), _ptr(cache.stats), rows // seq_len, seq_len, h, h_kv, dh,
            cache.key.shape[1], _ptr(seq_pos), n_split, _ptr(workspace), _ptr(out), _stream()), "attn_cached_ragged_int8")
        return out
    check(lib().ohara_attn_cached_int8(
        _ptr(q), _ptr(cache.key), _ptr(cache.value), _ptr(cache.stats), rows // seq_len, seq_len, h, h_kv, dh,
        cache.key.shape[1], int(pos), _ptr(pos_dev), n_split, _ptr(workspace), _ptr(out), _stream()), "attn_cached_int8")
    return out


def attn_decode(q, kcache, vcache, h, h_kv, dh, length, n_split, workspace, out=None, pos_dev=None):
    """Decode case: one query per sequence seeing `length` cached positions."""
    return attn_cached(q, kcache, vcache, h, h_kv, dh, length - 1, n_split, workspace, out, pos_dev, 1)


def advance_positions(seq_pos: torch.Tensor, active: torch.Tensor | None = None, by: int = 1) -> None:
    """seq_pos[b] += by where active[b] (uint8) is non-zero; all entries when ``active`` is None."""
    _need(seq_pos, torch.int32, "seq_pos")
    if active is not None:
        _need(active, torch.uint8, "active")
    check(lib().ohara_advance_positions(_ptr(seq_pos), _ptr(active), seq_pos.numel(), by, _stream()), "advance_positions")


def advance_ragged(seq_pos: torch.Tensor, active: torch.Tensor | None, new_ids: torch.Tensor, next_ids: torch.Tensor,
                   by: int = 1) -> None:
    """``advance_positions`` and, in the same launch, next_ids[b] = new_ids[b] where active[b], else 0."""
    _need(seq_pos, torch.int32, "seq_pos")
    _need(new_ids, torch.int64, "new_ids")
    _need(next_ids, torch.int64, "next_ids")
    if active is not None:
        _need(active, torch.uint8, "active")
    if new_ids.numel() != seq_pos.numel() or next_ids.numel() != seq_pos.numel():
        raise ValueError("one id per sequence is required")
    check(lib().ohara_advance_ragged(_ptr(seq_pos), _ptr(active), _ptr(new_ids), _ptr(next_ids), seq_pos.numel(), by,
                                     _stream()), "advance_ragged")


def set_slots(slots: list[int], positions: list[int] | None, seq_pos: torch.Tensor, active: torch.Tensor, next_ids: torch.Tensor,
              ids: torch.Tensor | None = None) -> None:
    """In one launch: seq_pos[slots[i]] = positions[i], active[slots[i]] = 1 and, with ``ids``, next_ids[slots[i]] = ids[i]; without
    ``positions`` the slots are left: all three 0."""
    _need(seq_pos, torch.int32, "seq_pos")
    _need(active, torch.uint8, "active")
    _need(next_ids, torch.int64, "next_ids")
    if ids is not None:
        _need(ids, torch.int64, "ids")
    n = len(slots)
    if active.numel() != seq_pos.numel() or next_ids.numel() != seq_pos.numel() or any(len(t) != n for t in (positions, ids) if t is not None):
        raise ValueError("one position and id per slot are required")
    check(lib().ohara_set_slots((C.c_int32 * n)(*slots), None if positions is None else (C.c_int32 * n)(*positions), n, int(positions is not None),
                                _ptr(ids), _ptr(next_ids), _ptr(seq_pos), _ptr(active), seq_pos.numel(), _stream()), "set_slots")


_zero_draws: dict = {}  # (rows, device) -> fp32 zeros


def argmax(logits: torch.Tensor, valid_vocab: int | None = None, next_ids=None, history=None, step_state=None):
    b, v = logits.shape
    if next_ids is None:
        next_ids = torch.empty(b, dtype=torch.int64, device=logits.device)
    if logits.dtype == torch.float32:
        # the candidates of top-k 1 are the ids tied at the maximum; a draw of 0 takes the lowest of them
        u = _zero_draws.get((b, logits.device))
        if u is None:
            u = _zero_draws[(b, logits.device)] = torch.zeros(b, dtype=torch.float32, device=logits.device)
        return sample_topk_topp(logits, 1.0, 1, 1.0, u, valid_vocab, out=next_ids, history=history, step_state=step_state)
    _need(logits, BF16, "logits")
    check(
        lib().ohara_argmax_bf16(
            _ptr(logits), logits.stride(0), b, v, v if valid_vocab is None else valid_vocab, _ptr(next_ids),
            _ptr(history), 0 if history is None else history.shape[0], _ptr(step_state), _stream(),
        ),
        "argmax",
    )
    return next_ids


def sample_topk_topp(logits: torch.Tensor, temperature: float, top_k: int, top_p: float, u: torch.Tensor,
                     valid_vocab: int | None = None, out=None, history=None, step_state=None,
                     u_per_step: bool = False, exclusive: bool = False, workspace=None) -> torch.Tensor:
    """logits (B, V) bf16 or fp32 on the device, u (B,) fp32 uniform draws -> ids (B,) int64.
    With ``u_per_step`` (needs step_state) u is (steps, B) and row ``step`` is read on the device.
    ``exclusive``: the caller's sampler calls on this GPU do not overlap in time (a decode loop on one
    stream), which lets a small top-k on a long row run on several workgroups (same results).
    ``workspace`` (``sample_workspace``): the same with the workgroups meeting in the caller's buffer instead of
    the library's, so that callers with a workspace each may overlap (one per decode session)."""
    if logits.dtype not in (BF16, torch.float32):
        raise ValueError("logits must be bfloat16 or float32")
    _need(logits, logits.dtype, "logits")
    _need(u, torch.float32, "u")
    b, v = logits.shape
    if u_per_step:
        if step_state is None or u.ndim != 2 or u.shape[1] != b:
            raise ValueError("u_per_step needs step_state and a (steps, batch) tensor of draws")
    elif u.numel() != b:
        raise ValueError("one uniform draw per row is required")
    if out is None:
        out = torch.empty(b, dtype=torch.int64, device=logits.device)
    args = (_ptr(logits), 1 if logits.dtype == torch.float32 else 0, logits.stride(0), b, v,
            v if valid_vocab is None else valid_vocab, float(temperature), int(top_k), float(top_p), _ptr(u),
            b if u_per_step else 0, _ptr(out), _ptr(history), 0 if history is None else history.shape[0], _ptr(step_state))
    if workspace is not None:
        _need(workspace, torch.uint8, "workspace")
        check(lib().ohara_sample_topk_topp_ws(*args, _ptr(workspace), workspace.numel(), _stream()), "sample_topk_topp")
        return out
    check((lib().ohara_sample_topk_topp_exclusive if exclusive else lib().ohara_sample_topk_topp)(*args, _stream()),
          "sample_topk_topp")
    return out


def sample_workspace(device) -> torch.Tensor:
    """A zeroed workspace for ``sample_topk_topp(..., workspace=)``: one per caller whose calls may overlap others'."""
    return torch.zeros(lib().ohara_sample_workspace_bytes(), dtype=torch.uint8, device=device)


# ---- BitLinear ---------------------------------------------------------------------------------


class PackedTernary:
    """Ternary weight (N, K) in the kernels' 2-bit layout with its per-tensor scale."""

    __slots__ = ("data", "n", "k", "gamma")

    def __init__(self, data, n, k, gamma):
        self.data, self.n, self.k, self.gamma = data, n, k, float(gamma)


def pack_ternary(t: torch.Tensor, gamma: float) -> PackedTernary:
    _need(t, torch.int8, "t")
    n, k = t.shape
    nbytes = C.c_int64(0)
    check(lib().ohara_bitlinear_pack_ternary(0, n, k, k, 0, C.byref(nbytes), 0), "pack_ternary size")
    dst = torch.empty(nbytes.value // 4, dtype=torch.int32, device=t.device)
    check(lib().ohara_bitlinear_pack_ternary(_ptr(t), n, k, k, _ptr(dst), None, _stream()), "pack_ternary")
    return PackedTernary(dst, n, k, gamma)


def act_quant(x: torch.Tensor, norm_w: torch.Tensor, eps: float = 1e-5):
    """(rows, K) bf16 -> q int8 (rows, K padded to 16), s fp32 (rows,), sum q int32 (rows,)."""
    _need(x, BF16, "x")
    rows, k = x.shape
    ldq = (k + 15) // 16 * 16
    q = torch.zeros(rows, ldq, dtype=torch.int8, device=x.device)
    s = torch.empty(rows, dtype=torch.float32, device=x.device)
    sq = torch.empty(rows, dtype=torch.int32, device=x.device)
    check(lib().ohara_act_quant_int8(_ptr(x), x.stride(0), _ptr(norm_w), eps, rows, k, _ptr(q), ldq, _ptr(s), _ptr(sq),
                                     _stream()), "act_quant")
    return q, s, sq


def gemv_ternary(q, s, sumq, w: PackedTernary, residual=None, out=None, want_acc=False):
    rows = q.shape[0]
    if out is None:
        out = torch.empty(rows, w.n, dtype=BF16, device=q.device)
    acc = torch.empty(rows, w.n, dtype=torch.int32, device=q.device) if want_acc else None
    check(lib().ohara_gemv_ternary_i8(_ptr(q), q.stride(0), _ptr(s), _ptr(sumq), _ptr(w.data), w.n, w.k, w.gamma, rows,
                                      _ptr(residual), 0 if residual is None else residual.stride(0), _ptr(out),
                                      out.stride(0), _ptr(acc), w.n, _stream()), "gemv_ternary")
    return (out, acc) if want_acc else out


# Rows up to which every workgroup of the fused BitLinear kernels quantises them in its own LDS; more are quantised once, then
# multiplied in tiles.  us of a layer's four calls, fused / tiles, captured: width 2048 8 rows 69 / 56, 12 92 / 57, 16 114 / 57, 64 551 / 62;
# 256 8 rows 26 / 27, 12 31 / 27, 64 118 / 32.  Launched one by one the tiles' ten launches a layer take the host 112 us, so that a
# whole prompt of the 24-layer model takes 2.6 / 2.9 ms at 12 rows, 3.2 / 2.9 at 16, 14.7 / 2.8 at 64.
BIT_ROWS = 12


def act_quant_sets(x, norm_ws, eps, pre_norm_w=None):
    """Codes of x (rows, K) for each norm weight (at most three): q (sets, rows, K padded to 16), s and sum q (sets, rows)."""
    _need(x, BF16, "x")
    rows, k = x.shape
    n, ldq = len(norm_ws), (k + 15) // 16 * 16
    q = torch.empty(n, rows, ldq, dtype=torch.int8, device=x.device)
    s = torch.empty(n, rows, dtype=torch.float32, device=x.device)
    sq = torch.empty(n, rows, dtype=torch.int32, device=x.device)
    nw = (C.c_void_p * n)(*[w.data_ptr() for w in norm_ws])
    check(lib().ohara_act_quant_sets_int8(_ptr(x), x.stride(0), _ptr(pre_norm_w), nw, n, eps, rows, k, _ptr(q), ldq, _ptr(s),
                                          _ptr(sq), _stream()), "act_quant_sets")
    return q, s, sq


def bitlinear_swiglu(gate, up, norm_w, w: PackedTernary, eps=1e-5, residual=None):
    """BitLinear on rows silu(gate) * up (rows, K) each, quantised as they are multiplied out, in tiles."""
    _need(gate, BF16, "gate")
    _need(up, BF16, "up")
    rows, k = gate.shape
    if k != w.k or up.shape != gate.shape:
        raise ValueError(f"gate and up have {k} and {up.shape[1]} columns, weight expects {w.k}")
    ldq = (k + 15) // 16 * 16
    q = torch.empty(rows, ldq, dtype=torch.int8, device=gate.device)
    s = torch.empty(rows, dtype=torch.float32, device=gate.device)
    sq = torch.empty(rows, dtype=torch.int32, device=gate.device)
    check(lib().ohara_act_quant_swiglu_int8(_ptr(gate), _ptr(up), k, _ptr(norm_w), eps, rows, k, _ptr(q), ldq, _ptr(s), _ptr(sq), _stream()),
          "act_quant_swiglu")
    return gemv_ternary(q, s, sq, w, residual)


def bitlinear_many(x, pre_norm_w, projs, eps=1e-5):
    """Several BitLinears of one width on the same rows (any number), each row quantised once for each -> their outputs.
    ``projs``: at most three (norm_w, PackedTernary) pairs."""
    n, rows, width = len(projs), x.shape[0], projs[0][1].n
    if any(w.n != width or w.k != x.shape[1] for _, w in projs):
        raise ValueError(f"x has {x.shape[1]} columns, weights expect {[w.k for _, w in projs]} and give {[w.n for _, w in projs]}")
    q, s, sq = act_quant_sets(x, [p[0] for p in projs], eps, pre_norm_w)
    outs = [torch.empty(rows, width, dtype=BF16, device=x.device) for _ in projs]
    wp = (C.c_void_p * n)(*[p[1].data.data_ptr() for p in projs])
    gm = (C.c_float * n)(*[p[1].gamma for p in projs])
    check(lib().ohara_gemm_ternary_sets_i8(_ptr(q), q.stride(1), _ptr(s), _ptr(sq), wp, gm, n, width, x.shape[1], rows,
                                           (C.c_void_p * n)(*[t.data_ptr() for t in outs]), width, _stream()), "gemm_ternary_sets")
    return outs


def bitlinear(x, norm_w, w: PackedTernary, eps=1e-5, residual=None, out=None, want_acc=False, pre_norm_w=None):
    """Fused BitLinear.forward on rows of x (rows, K) bf16; ``pre_norm_w`` applies a block-level
    RMSNorm to x first, in the same pass."""
    _need(x, BF16, "x")
    rows, k = x.shape
    if k != w.k:
        raise ValueError(f"x has {k} columns, weight expects {w.k}")
    if out is None:
        out = torch.empty(rows, w.n, dtype=BF16, device=x.device)
    if rows > BIT_ROWS:
        q, s, sq = act_quant_sets(x, [norm_w], eps, pre_norm_w)
        return gemv_ternary(q[0], s[0], sq[0], w, residual, out, want_acc)
    acc = torch.empty(rows, w.n, dtype=torch.int32, device=x.device) if want_acc else None
    check(lib().ohara_bitlinear_bf16(_ptr(x), x.stride(0), _ptr(pre_norm_w), _ptr(norm_w), eps, _ptr(w.data), w.n, w.k, w.gamma, rows,
                                     _ptr(residual), 0 if residual is None else residual.stride(0), _ptr(out),
                                     out.stride(0), _ptr(acc), w.n, _stream()), "bitlinear")
    return (out, acc) if want_acc else out


def bitlinear_qkv_rope_append(x, pre_norm_w, projs, eps, h, h_kv, dh, cos, sin, pos, kcache, vcache, q_out=None,
                              pos_dev=None, seq_len=1):
    """The query / key / value BitLinears of one layer on rows of x in one launch (more than BIT_ROWS rows: behind one that quantises
    them), with rotary + cache append.  ``projs``: three (norm_w, PackedTernary) pairs.  Returns q (rows, h*dh)."""
    _need(x, BF16, "x")
    rows, k = x.shape
    if q_out is None:
        q_out = torch.empty(rows, h * dh, dtype=BF16, device=x.device)
    nw = (C.c_void_p * 3)(*[p[0].data_ptr() for p in projs])
    wp = (C.c_void_p * 3)(*[p[1].data.data_ptr() for p in projs])
    gm = (C.c_float * 3)(*[p[1].gamma for p in projs])
    if rows > BIT_ROWS:
        if any(w.k != k or w.n != heads * dh for (_, w), heads in zip(projs, (h, h_kv, h_kv))):
            raise ValueError(f"x has {k} columns and heads are {h}, {h_kv} x {dh}, weights expect {[w.k for _, w in projs]} and give {[w.n for _, w in projs]}")
        q, s, sq = act_quant_sets(x, [p[0] for p in projs], eps, pre_norm_w)
        check(lib().ohara_gemm_ternary_qkv_rope_append(
            _ptr(q), q.stride(1), _ptr(s), _ptr(sq), wp, gm, k, rows // seq_len, seq_len, h, h_kv, dh, _ptr(cos), _ptr(sin),
            int(pos), _ptr(pos_dev), _ptr(q_out), _ptr(kcache), _ptr(vcache), kcache.shape[1], _stream()),
            "gemm_ternary_qkv_rope_append")
        return q_out
    check(lib().ohara_bitlinear_qkv_rope_append_bf16(
        _ptr(x), x.stride(0), _ptr(pre_norm_w), eps, k, nw, wp, gm, rows // seq_len, seq_len, h, h_kv, dh, _ptr(cos),
        _ptr(sin), int(pos), _ptr(pos_dev), _ptr(q_out), _ptr(kcache), _ptr(vcache), kcache.shape[1], _stream()),
        "bitlinear_qkv_rope_append")
    return q_out


def bitlinear_gate_up(x, pre_norm_w, gate, up, eps=1e-5, out=None):
    """silu(gate(x)) * up(x) for two BitLinears ((norm_w, PackedTernary) pairs) on rows of x (<= 64)."""
    _need(x, BF16, "x")
    rows, k = x.shape
    f = gate[1].n
    if out is None:
        out = torch.empty(rows, f, dtype=BF16, device=x.device)
    check(lib().ohara_bitlinear_gate_up_bf16(
        _ptr(x), x.stride(0), _ptr(pre_norm_w), eps, k, f, _ptr(gate[0]), _ptr(gate[1].data), gate[1].gamma,
        _ptr(up[0]), _ptr(up[1].data), up[1].gamma, rows, _ptr(out), out.stride(0), _stream()), "bitlinear_gate_up")
    return out


def silu_mul(gate, up, out=None):
    _need(gate, BF16, "gate")
    _need(up, BF16, "up")
    if out is None:
        out = torch.empty_like(gate)
    check(lib().ohara_silu_mul_bf16(_ptr(gate), _ptr(up), _ptr(out), gate.numel(), _stream()), "silu_mul")
    return out


def rope_append(q, k, v, batch, seq_len, h, h_kv, dh, cos, sin, pos, kcache, vcache, pos_dev=None):
    """In-place rotary on q (rows, h*dh); rotated k and v appended to the cache."""
    check(lib().ohara_rope_append_bf16(_ptr(q), _ptr(k), _ptr(v), batch, seq_len, h, h_kv, dh, _ptr(cos), _ptr(sin),
                                       int(pos), _ptr(pos_dev), _ptr(kcache), _ptr(vcache), kcache.shape[1], _stream()),
          "rope_append")
    return q


def rope_rows(q, k, v, batch, seq_len, h, h_kv, dh, cos, sin, pos, pos_dev=None):
    """In-place rotary on q; returns the rotated k and v as (batch, seq_len, h_kv, dh) tensors (what an int8
    cache's append quantises)."""
    kr, vr = torch.empty_like(k), torch.empty_like(v)
    check(lib().ohara_rope_append_bf16(_ptr(q), _ptr(k), _ptr(v), batch, seq_len, h, h_kv, dh, _ptr(cos), _ptr(sin),
                                       int(pos), _ptr(pos_dev), _ptr(kr), _ptr(vr), 0, _stream()), "rope_rows")
    return kr.view(batch, seq_len, h_kv, dh), vr.view(batch, seq_len, h_kv, dh)


# ---- Phi (ohara/models/phi.py) ----------------------------------------------------------------

_LIN_EPI = {"bias": 0, "gelu": 1, "add2": 2}


def linear_bias(x, w: PackedLinear, bias, epilogue: str = "bias", add1=None, add2=None, out=None) -> torch.Tensor:
    """nn.Linear with bias on a packed weight; ``epilogue``: "bias", "gelu" (new_gelu of the result,
    phi.py:37-40) or "add2" (bf16(bf16(add1 + y) + add2), phi.py:151).  x: (rows, K), any row stride."""
    if x.dtype != BF16 or not x.is_cuda or x.stride(1) != 1:
        raise ValueError("x must be a bf16 device matrix with unit column stride")
    _need(bias, BF16, "bias")
    rows, k = x.shape
    if k != w.k or bias.numel() != w.n:
        raise ValueError(f"x has {k} columns / bias {bias.numel()} entries, weight is {w.n} x {w.k}")
    if out is None:
        out = torch.empty(rows, w.n, dtype=BF16, device=x.device)
    for t in (add1, add2):
        if t is not None and (t.dtype != BF16 or t.stride(1) != 1):
            raise ValueError("addends must be bf16 with unit column stride")
    if epilogue == "add2" and add1 is not None and add2 is not None:
        room = lib().ohara_linear_bias_add2_bytes(rows, w.n, w.k)
        if room > 0:  # few rows for the depth: a product in parts
            workspace = torch.empty(room, dtype=torch.uint8, device=x.device)
            check(lib().ohara_linear_bias_add2_bf16(
                _ptr(x), x.stride(0), _ptr(w.data), w.n, w.k, _ptr(bias), rows, _ptr(add1), add1.stride(0), _ptr(add2),
                add2.stride(0), _ptr(out), out.stride(0), _ptr(workspace), room, _stream()), "linear_bias")
            return out
    check(
        lib().ohara_linear_bias_bf16(
            _ptr(x), x.stride(0), _ptr(w.data), w.n, w.k, _ptr(bias), rows, _LIN_EPI[epilogue],
            _ptr(add1), 0 if add1 is None else add1.stride(0), _ptr(add2), 0 if add2 is None else add2.stride(0),
            _ptr(out), out.stride(0), _stream(),
        ),
        "linear_bias",
    )
    return out


def phi_block_norms(rows, d, ff) -> bool:
    """Whether ``phi_block_in`` on rows before their LayerNorm is quicker than ``layernorm`` ahead of it."""
    return bool(lib().ohara_phi_block_norms(rows, d, ff))


def phi_block_in(x, ln_w, ln_b, eps, w: PackedLinear, bias, d, ff, batch, seq_len, pos, kcache, vcache, q, act,
                 pos_dev=None) -> None:
    """LayerNorm + [q; k; v; fc1] projection with bias + cache append + new_gelu in one launch
    (phi.py:150, :81-87, :95, :50-51).  x: (rows, d); q: (rows, d); act: (rows, ff)."""
    _need(x, BF16, "x")
    if w.n != 3 * d + ff or w.k != d or bias.numel() != w.n:
        raise ValueError("packed weight / bias do not match [q; k; v; fc1]")
    check(lib().ohara_phi_block_in_bf16(_ptr(x), x.stride(0), _ptr(ln_w), _ptr(ln_b), eps, _ptr(w.data), _ptr(bias), d, ff,
                                        batch, seq_len, pos, _ptr(pos_dev), _ptr(q), q.stride(0), _ptr(kcache), _ptr(vcache),
                                        kcache.shape[1], _ptr(act), act.stride(0), _stream()), "phi_block_in")


def layernorm(x, weight, bias, eps: float = 1e-5, out=None) -> torch.Tensor:
    """nn.LayerNorm over the last dimension of a (rows, d) bf16 matrix (phi.py:132, :160)."""
    _need(x, BF16, "x")
    rows, d = x.shape
    if out is None:
        out = torch.empty_like(x)
    check(lib().ohara_layernorm_bf16(_ptr(x), x.stride(0), _ptr(weight), _ptr(bias), _ptr(out), out.stride(0), rows, d, eps,
                                     _stream()), "layernorm")
    return out


def kv_append(k, v, kcache, vcache, batch, seq_len, h, dh, pos, pos_dev=None) -> None:
    """Rows (b, s) of k / v (views with a common row stride) -> cache[b, pos + s] as they are
    (phi.py:95)."""
    if k.stride(0) != v.stride(0) or k.stride(1) != 1 or v.stride(1) != 1:
        raise ValueError("k and v must share a row stride and have unit column stride")
    check(lib().ohara_kv_append_bf16(_ptr(k), _ptr(v), k.stride(0), batch, seq_len, h, dh, pos, _ptr(pos_dev), _ptr(kcache),
                                     _ptr(vcache), kcache.shape[1], _stream()), "kv_append")


def phi_attn_workspace(batch, h, dh, n_split, device) -> torch.Tensor:
    nbytes = lib().ohara_phi_attn_workspace_bytes(batch, h, dh, n_split)
    if nbytes < 0:
        raise ValueError("phi_attn_workspace: invalid sizes")
    return torch.zeros(nbytes, dtype=torch.uint8, device=device)  # the chunk counters start at zero


def phi_attn(q, kcache, vcache, cos, sin, rot, batch, seq_len, h, dh, pos, pos_dev=None, out=None, n_split=1,
             workspace=None) -> torch.Tensor:
    """PhiMHA's attention core over the cache (phi.py:98-117); q: (rows, h*dh) view with any row
    stride; cos / sin: fp32 (t_max, rot/2).  ``n_split`` > 1 (single-token calls) spreads the context
    over that many workgroups per (sequence, head); ``workspace`` from ``phi_attn_workspace``."""
    if q.stride(1) != 1:
        raise ValueError("q must have unit column stride")
    if cos.dtype != torch.float32 or sin.dtype != torch.float32:
        raise ValueError("cos / sin must be fp32")
    if out is None:
        out = torch.empty(batch * seq_len, h * dh, dtype=BF16, device=q.device)
    check(lib().ohara_phi_attn_bf16(_ptr(q), q.stride(0), _ptr(kcache), _ptr(vcache), _ptr(cos), _ptr(sin), rot, batch,
                                    seq_len, h, dh, kcache.shape[1], pos, _ptr(pos_dev), n_split, _ptr(workspace), _ptr(out),
                                    _stream()), "phi_attn")
    return out


def phi_attn_linear(q, kcache, vcache, cos, sin, rot, batch, h, dh, pos, x, w: PackedLinear, bias, pos_dev=None, out=None, y=None, n_split=1,
                    workspace=None):
    """``phi_attn`` of one token a sequence and, beside it in the same launch, ``linear_bias(x, w, bias)`` -> (out, y)."""
    if q.stride(1) != 1:
        raise ValueError("q must have unit column stride")
    if cos.dtype != torch.float32 or sin.dtype != torch.float32:
        raise ValueError("cos / sin must be fp32")
    if x.dtype != BF16 or not x.is_cuda or x.stride(1) != 1:
        raise ValueError("x must be a bf16 device matrix with unit column stride")
    _need(bias, BF16, "bias")
    if x.shape != (batch, w.k) or bias.numel() != w.n:
        raise ValueError(f"x is {tuple(x.shape)} / bias {bias.numel()} entries, weight is {w.n} x {w.k}")
    if out is None:
        out = torch.empty(batch, h * dh, dtype=BF16, device=q.device)
    if y is None:
        y = torch.empty(batch, w.n, dtype=BF16, device=q.device)
    check(lib().ohara_phi_attn_linear_bf16(_ptr(q), q.stride(0), _ptr(kcache), _ptr(vcache), _ptr(cos), _ptr(sin), rot, batch, h, dh, kcache.shape[1],
                                           pos, _ptr(pos_dev), n_split, _ptr(workspace), _ptr(out), _ptr(x), x.stride(0), _ptr(w.data), w.n, w.k,
                                           _ptr(bias), _ptr(y), y.stride(0), _stream()), "phi_attn_linear")
    return out, y


def phi_attn_out_chunks(batch, h, dh, rot, n_split, pos, n, k) -> int:
    """Chunks of a context at most in ``phi_attn_out``; 0 where that call is refused."""
    return lib().ohara_phi_attn_out_chunks(batch, h, dh, rot, n_split, pos, n, k)


def phi_attn_out(q, kcache, vcache, cos, sin, rot, batch, h, dh, pos, x, w: PackedLinear, bias, pos_dev, y, n_split, workspace, w_out: PackedLinear,
                 bias_out, add, out) -> torch.Tensor:
    """``phi_attn_linear`` and then ``linear_bias(attention, w_out, bias_out, "add2", add1=y, add2=add)``, whose launch merges the attention's chunks."""
    if q.stride(1) != 1:
        raise ValueError("q must have unit column stride")
    if cos.dtype != torch.float32 or sin.dtype != torch.float32:
        raise ValueError("cos / sin must be fp32")
    for t, name, width in ((x, "x", w.k), (y, "y", w.n), (add, "add", w.n), (out, "out", w.n)):
        if t.dtype != BF16 or not t.is_cuda or t.stride(1) != 1 or t.shape != (batch, width):
            raise ValueError(f"{name} must be a bf16 device matrix ({batch}, {width}) with unit column stride")
    if w_out.n != w.n or w_out.k != h * dh or bias.numel() != w.n or bias_out.numel() != w.n:
        raise ValueError(f"weights are {w.n} x {w.k} and {w_out.n} x {w_out.k} with {bias.numel()} and {bias_out.numel()} biases, heads {h} x {dh}")
    check(lib().ohara_phi_attn_out_bf16(_ptr(q), q.stride(0), _ptr(kcache), _ptr(vcache), _ptr(cos), _ptr(sin), rot, batch, h, dh, kcache.shape[1], pos,
                                        _ptr(pos_dev), n_split, _ptr(workspace), _ptr(x), x.stride(0), _ptr(w.data), w.n, w.k, _ptr(bias), _ptr(y),
                                        y.stride(0), _ptr(w_out.data), _ptr(bias_out), _ptr(add), add.stride(0), _ptr(out), out.stride(0), _stream()),
          "phi_attn_out")
    return out


# ---- hybrid decoders: attention with a distance bias beside recurrent layers -------------------------
# bf16 or fp32 activations: the entry point follows the dtype of the activations.

F32 = torch.float32


def _typed(name: str, dtype):
    return getattr(lib(), f"ohara_{name}_{'f32' if dtype == F32 else 'bf16'}")


def round8(n: int) -> int:
    return (n + 7) // 8 * 8


class Seq:
    """Which rows of a call belong to which sequence and where they sit (OharaSeq).  ``pos_dev`` (int32): one
    position for all sequences, or one per sequence with ``per_sequence``; ``lens`` / ``slots`` (int32, one entry per
    sequence): tokens of each sequence in the call, cache row of each sequence."""

    __slots__ = ("c", "batch", "seq_len", "lens", "host", "carry", "_keep")

    def __init__(self, batch: int, seq_len: int, pos: int = 0, pos_dev=None, per_sequence: bool = False, lens=None, slots=None,
                 host=None):
        """``host``: (starts, counts, rows of the cache) of the sequences as lists, where the caller knows them.  ``carry``: what layers
        leave to later layers of the same call."""
        for name, t in (("pos_dev", pos_dev), ("lens", lens), ("slots", slots)):
            if t is not None:
                _need(t, torch.int32, name)
                if t.numel() < (1 if name == "pos_dev" and not per_sequence else batch):
                    raise ValueError(f"{name}: one entry per sequence is required")
        self.batch, self.seq_len, self.lens, self.host = batch, seq_len, lens, host
        self._keep, self.carry = (pos_dev, lens, slots), {}
        self.c = _lib.OharaSeq(batch, seq_len, int(pos), int(per_sequence), _ptr(pos_dev), _ptr(lens), _ptr(slots))

    @property
    def pos_dev(self):
        return self._keep[0]

    @property
    def rows(self) -> int:
        return self.batch * self.seq_len

    @property
    def ref(self):
        return C.byref(self.c)


class Mixture:
    """What routed experts leave to be summed (OharaMixture): row n of the layer's output is sum_j w[n, j] * (y[pos_of[n, j]], or h[n]
    where idx[n, j] names an identity output) + shared[n]; w None: all weights are 1."""

    __slots__ = ("c", "_keep")

    def __init__(self, idx, w, pos_of, y, h, shared, experts: int):
        self._keep = (idx, w, pos_of, y, h, shared)
        self.c = _lib.OharaMixture(idx.shape[1], experts, y.stride(0), h.stride(0), 0 if shared is None else shared.stride(0), 0, _ptr(w),
                                   _ptr(idx), _ptr(pos_of), _ptr(y), _ptr(h), _ptr(shared))

    @property
    def dtype(self):
        return self._keep[3].dtype


def residual_norm(x, seq: Seq, dtype, *, ids=None, table=None, table_scale=1.0, y=None, mix: Mixture | None = None, norm_w=None, groups=1,
                  eps=0.0, mode="none", norm2_w=None, conv_w=None, ring=None, center_y=False, center_out=False):
    """x (rows, d) fp32 <- table_scale * table[ids], or x + norm_w * group_rms(y) (``mix``: of a mixture of experts; without norm_w: x + y), in place; returns
    what ``mode`` asks for as (rows, d rounded up to 8) in ``dtype``: "copy" of x, "conv" (x + causal depthwise convolution over time, one token per
    sequence, ring updated), "norm" (group RMS norm of x times norm2_w), or None.  ``center_y`` / ``center_out``: the norm
    of y / of the output is a layer norm without bias."""
    _need(x, F32, "x")
    rows, d = x.shape
    m = {"none": _lib.OUT_NONE, "copy": _lib.OUT_COPY, "conv": _lib.OUT_CONV, "norm": _lib.OUT_NORM}[mode]
    m |= (_lib.CENTER_Y if center_y else 0) | (_lib.CENTER_OUT if center_out else 0)
    if rows != seq.rows:
        raise ValueError("x has one row per token of the call")
    for t, name in ((y, "y"), (table, "table")):
        if t is not None:
            _need(t, dtype, name)
    if mix is not None and mix.dtype != dtype:
        raise ValueError("the mixture is of another dtype")
    out = torch.empty(rows, round8(d), dtype=dtype, device=x.device) if mode != "none" else None
    check(_typed("residual_norm", dtype)(
        _ptr(x), d, _ptr(ids), _ptr(table), 0 if table is None else table.shape[0], table_scale, _ptr(y),
        0 if y is None else y.stride(0), _ptr(norm_w), groups, eps, m, _ptr(out), 0 if out is None else out.stride(0), _ptr(norm2_w), _ptr(conv_w),
        0 if conv_w is None else conv_w.shape[0], _ptr(ring), None if mix is None else C.byref(mix.c), seq.ref, _stream()), "residual_norm")
    return out


def input_conv(x, conv_w, ring, seq: Seq, dtype):
    """x (rows, d) fp32 -> x + causal depthwise convolution over time, (rows, d rounded up to 8) in ``dtype``; then the
    last inputs of every sequence go into the ring."""
    _need(x, F32, "x")
    rows, d = x.shape
    taps = conv_w.shape[0]
    out = torch.empty(rows, round8(d), dtype=dtype, device=x.device)
    check(_typed("input_conv", dtype)(_ptr(x), d, _ptr(conv_w), taps, _ptr(ring), _ptr(out), out.stride(0), seq.ref, _stream()),
          "input_conv")
    conv_ring_store(x, d, ring, seq)
    return out


def conv_ring_store(src, channels: int, ring, seq: Seq) -> None:
    """The last inputs of every sequence (the first ``channels`` columns of src) -> ring (cache rows, taps, channels)."""
    if ring.shape[2] != channels or ring.dtype != src.dtype or src.shape[0] != seq.rows:
        raise ValueError("ring does not fit the inputs")
    check(_typed("conv_ring_store", src.dtype)(_ptr(src), src.stride(0), channels, ring.shape[1], _ptr(ring), seq.ref, _stream()),
          "conv_ring_store")


def gemm_f32(x, w, bias=None, w_up=None, cap: float = 0.0, out=None):
    """fp32 y = x W^T (+ bias, cap * tanh(y / cap)), or silu(x W^T) * (x w_up^T).  x: (rows, K), any row stride."""
    if x.dtype != F32 or not x.is_cuda or x.stride(1) != 1 or x.shape[1] != w.shape[1]:
        raise ValueError("x must be an fp32 device matrix with unit column stride and W's columns")
    rows, n = x.shape[0], w.shape[0]
    if out is None:
        out = torch.empty(rows, n, dtype=F32, device=x.device)
    check(lib().ohara_gemm_f32(_ptr(x), x.stride(0), _ptr(w), _ptr(w_up), _ptr(bias), cap, n, w.shape[1], rows, _ptr(out),
                               out.stride(0), _stream()), "gemm_f32")
    return out


def gemm_xielu(x, w, bias, above: float, below: float, out=None):
    """z / 2 + (above z^2 if z > 0 else below (exp(z) - 1 - z)), z = x W^T + bias; w: packed (bf16) or (n, k) fp32."""
    f32 = x.dtype == F32
    n, k = w.shape if f32 else (w.n, w.k)
    if not x.is_cuda or x.stride(1) != 1 or x.shape[1] != k or bias.numel() != n or bias.dtype != x.dtype:
        raise ValueError("x must be a device matrix with unit column stride and W's columns, bias W's rows")
    if out is None:
        out = torch.empty(x.shape[0], n, dtype=x.dtype, device=x.device)
    check(_typed("gemm_xielu", x.dtype)(_ptr(x), x.stride(0), _ptr(w if f32 else w.data), n, k, _ptr(bias), above, below, x.shape[0],
                                        _ptr(out), out.stride(0), _stream()), "gemm_xielu")
    return out


def gemm_softcap(x, w: PackedLinear, cap: float, out=None):
    """bf16(cap * tanh(x W^T / cap)) on a packed weight."""
    _need(x, BF16, "x")
    rows, k = x.shape
    if k != w.k:
        raise ValueError(f"x has {k} columns, weight expects {w.k}")
    if out is None:
        out = torch.empty(rows, w.n, dtype=BF16, device=x.device)
    check(lib().ohara_gemm_softcap_bf16(_ptr(x), x.stride(0), _ptr(w.data), w.n, w.k, cap, rows, _ptr(out), out.stride(0),
                                        _stream()), "gemm_softcap")
    return out


def gemm_gelu_lookup(x, w, table, column: int, ids, out=None):
    """gelu_tanh(x W^T) * table[ids, column: column + n]; w: a packed weight (bf16) or (n, k) fp32, table (vocab, columns), ids
    (rows,) int64 on the device."""
    f32 = x.dtype == F32
    n, k = w.shape if f32 else (w.n, w.k)
    if not x.is_cuda or x.stride(1) != 1 or x.shape[1] != k or table.dtype != x.dtype or not table.is_contiguous():
        raise ValueError("x and table must be device matrices of one dtype, x with W's columns")
    if column < 0 or column + n > table.shape[1] or ids.dtype != torch.int64 or ids.numel() != x.shape[0]:
        raise ValueError("the table has no such columns, or ids are not one int64 per row")
    if out is None:
        out = torch.empty(x.shape[0], n, dtype=x.dtype, device=x.device)
    check(_typed("gemm_gelu_lookup", x.dtype)(
        _ptr(x), x.stride(0), _ptr(w if f32 else w.data), n, k, _ptr(table) + column * table.element_size(), table.stride(0),
        _ptr(ids), table.shape[0], x.shape[0], _ptr(out), out.stride(0), _stream()), "gemm_gelu_lookup")
    return out


TOKEN_SIDE_ELEMENTS = 16384  # of the residual that a workgroup of token_side holds


def token_side(x, y, norm_w, gate: PackedLinear, proj: PackedLinear, table, column: int, ids, side_w, eps: float, out_w, *,
               center_y=False, center_out=False, rows_per_group: int | None = None):
    """x (rows, d) fp32 += norm_w * norm(y); x += side_w * rms(proj(gelu_tanh(gate x) * table[ids, column: column + n])); returns
    out_w * norm(x) as (rows, round8(d)) bf16.  One launch; d a multiple of 4."""
    _need(x, F32, "x")
    _need(y, BF16, "y")
    rows, d = x.shape
    if gate.k != round8(d) or proj.n != round8(d) or proj.k != gate.n or y.shape[0] != rows or ids.numel() != rows or ids.dtype != torch.int64:
        raise ValueError("token_side: operands do not fit the residual")
    if table.dtype != BF16 or not table.is_contiguous() or column < 0 or column + gate.n > table.shape[1]:
        raise ValueError("the table has no such columns")
    if rows_per_group is None:  # four, and more where that fills the 256 CUs more than once
        rows_per_group = 1
        while rows_per_group < 16 and 2 * rows_per_group * d <= TOKEN_SIDE_ELEMENTS and (rows_per_group < 4 or rows > 256 * rows_per_group):
            rows_per_group *= 2
    out = torch.empty(rows, round8(d), dtype=BF16, device=x.device)
    check(lib().ohara_token_side_bf16(
        _ptr(x), d, _ptr(y), y.stride(0), _ptr(norm_w), int(center_y), _ptr(gate.data), _ptr(proj.data), gate.n,
        _ptr(table) + column * table.element_size(), table.stride(0), _ptr(ids), table.shape[0], _ptr(side_w), eps, _ptr(out_w),
        int(center_out), rows, rows_per_group, _ptr(out), out.stride(0), _stream()), "token_side")
    return out


def qkv_rotate_append(p, h, h_kv, dh, dv, cos, sin, rot, kcache, vcache, seq: Seq):
    """p rows [q; k; v; ...] -> q (rows, h * round8(dh)); keys and values into the caches; the first ``rot`` dimensions of q and
    k heads rotated in neighbouring pairs by the tables cos, sin (positions, rot / 2) fp32."""
    if rot and (cos.shape != (cos.shape[0], rot // 2) or cos.shape[0] < kcache.shape[1] or cos.shape != sin.shape):
        raise ValueError("rotary tables must cover the cache's positions with rot / 2 angles each")
    q = torch.empty(p.shape[0], h * round8(dh), dtype=p.dtype, device=p.device)
    check(_typed("qkv_rotate_append", p.dtype)(
        _ptr(p), p.stride(0), h, h_kv, dh, dv, _ptr(cos), _ptr(sin), rot, _ptr(q), _ptr(kcache), _ptr(vcache), kcache.shape[1],
        seq.ref, _stream()), "qkv_rotate_append")
    return q


def qkv_headnorm_rotate_append(p, h, h_kv, dh, dv, qn, kn, eps, cos, sin, rot, kcache, vcache, seq: Seq):
    """``qkv_rotate_append`` with every q and k head first over its own root mean square times qn / kn (dh entries, fp32)."""
    if rot and (cos.shape != (cos.shape[0], rot // 2) or cos.shape[0] < kcache.shape[1] or cos.shape != sin.shape):
        raise ValueError("rotary tables must cover the cache's positions with rot / 2 angles each")
    if qn.numel() != dh or kn.numel() != dh:
        raise ValueError("head norms have one weight per dimension of a head")
    q = torch.empty(p.shape[0], h * round8(dh), dtype=p.dtype, device=p.device)
    check(_typed("qkv_headnorm_rotate_append", p.dtype)(
        _ptr(p), p.stride(0), h, h_kv, dh, dv, _ptr(qn), _ptr(kn), eps, _ptr(cos), _ptr(sin), rot, _ptr(q), _ptr(kcache), _ptr(vcache),
        kcache.shape[1], seq.ref, _stream()), "qkv_headnorm_rotate_append")
    return q


def qkv_norm_append(p, h, h_kv, dh, dv, qn, kn, eps, kcache, vcache, seq: Seq):
    """p rows [q; k; v; ...] -> normalised q (rows, h * round8(dh)); keys and values into the caches."""
    q = torch.empty(p.shape[0], h * round8(dh), dtype=p.dtype, device=p.device)
    check(_typed("qkv_norm_append", p.dtype)(_ptr(p), p.stride(0), h, h_kv, dh, dv, _ptr(qn), _ptr(kn), eps, _ptr(q), _ptr(kcache),
                                             _ptr(vcache), kcache.shape[1], seq.ref, _stream()), "qkv_norm_append")
    return q


def attn_bias_workspace(rows, h, dv, n_split, device) -> torch.Tensor:
    n = lib().ohara_attn_bias_workspace_bytes(rows, h, dv, n_split)
    if n < 0:
        raise ValueError("bad attention workspace shape")
    return torch.zeros(n, dtype=torch.uint8, device=device)  # the chunk counters start at zero


def attn_bias(q, kcache, vcache, h, h_kv, dh, dv, scale, slopes, gate, seq: Seq, n_split=1, workspace=None):
    """Causal attention with the bias -slopes[head] * distance, head outputs times sigmoid(gate) -> (rows, round8(h * dv)).
    gate: a (rows, h) column slice of the projection (or None)."""
    out = torch.empty(q.shape[0], round8(h * dv), dtype=q.dtype, device=q.device)
    check(_typed("attn_bias", q.dtype)(
        _ptr(q), _ptr(kcache), _ptr(vcache), h, h_kv, dh, dv, kcache.shape[1], scale, _ptr(slopes), _ptr(gate),
        0 if gate is None else gate.stride(0), n_split, _ptr(workspace), _ptr(out), out.stride(0), seq.ref, _stream()),
        "attn_bias")
    return out


def attn_scored(q, keys, values, h, h_kv, dh, dv, t_max, scale, seq: Seq, *, cap=0.0, chunk=0, window=0, sinks=None, slopes=None,
                gate=None, gate_elements=False, ld_k=0, ld_v=0, n_split=1, workspace=None, out_scale=1.0, out=None, k_shared=None, ld_shared=0,
                d_shared=0):
    """Causal attention over positions of ``keys`` / ``values`` (cache rows of t_max positions, ``ld_k`` / ``ld_v`` elements apart if
    not densely packed) -> (rows, round8(h * dv)).  Scores: scale q . k, soft-capped by ``cap``, minus slopes[head] * distance;
    ``chunk``: inside chunks of that many positions.  gate: a (rows, h) or, ``gate_elements``, (rows, h * dv) column slice,
    through the sigmoid.  ``window``: only that many keys up to the query's own; ``sinks`` (h,) fp32: scores that join the softmax
    without a value.  ``out``: a column slice of a wider buffer.  ``k_shared``: the last ``d_shared`` elements of every head's keys,
    ``ld_shared`` elements between positions.  q may be the first columns of wider rows."""
    if out is None:
        out = torch.empty(q.shape[0], round8(h * dv), dtype=q.dtype, device=q.device)
    elif out.shape != (q.shape[0], round8(h * dv)) or out.dtype != q.dtype or out.stride(1) != 1:
        raise ValueError("out must be (rows, round8(h * dv)) with unit column stride")
    sc = _lib.OharaScores(scale, cap, chunk, int(gate_elements), ld_k, ld_v, _ptr(slopes), _ptr(sinks), window, out_scale,
                          _ptr(k_shared), ld_shared, d_shared, q.stride(0), 0)
    check(_typed("attn_scored", q.dtype)(
        _ptr(q), _ptr(keys), _ptr(values), h, h_kv, dh, dv, t_max, C.byref(sc), _ptr(gate), 0 if gate is None else gate.stride(0),
        n_split, _ptr(workspace), _ptr(out), out.stride(0), seq.ref, _stream()), "attn_scored")
    return out


def attn_mixed_workspace(batch, seq_len, h, h_kv, dh, dv, positions, window, keep, n_split, dtype, device) -> torch.Tensor:
    n = lib().ohara_attn_mixed_workspace_bytes(batch, seq_len, h, h_kv, dh, dv, positions, window, keep, n_split, 4 if dtype == F32 else 2)
    if n < 0:
        raise ValueError("bad attention workspace shape")
    make = torch.zeros if seq_len == 1 else torch.empty  # the chunk counters of a decode step start at zero
    return make(n, dtype=torch.uint8, device=device)


def attn_mixed(q, kcache, vcache, h, h_kv, dh, dv, scale, talk, seq: Seq, *, temp=None, window=0, keep=0, positions=None, n_split=1,
               workspace=None):
    """Causal attention whose softmax weights are mixed across heads by talk (h, h) fp32 before they meet the values -> (rows,
    round8(h * dv)).  temp (h,) fp32: factors of the scores.  ``window`` > 0: that many keys up to the query's own, and the ``keep``
    first positions.  ``positions``: no sequence ends past it (None: the caches' capacity)."""
    t_max = kcache.shape[1]
    positions = t_max if positions is None else positions
    for t, n, name in ((talk, h * h, "talk"), (temp, h, "temp")):
        if t is not None and (t.dtype != F32 or t.numel() != n or not t.is_contiguous()):
            raise ValueError(f"{name} must hold {n} fp32 values")
    if workspace is None:
        workspace = attn_mixed_workspace(seq.batch, seq.seq_len, h, h_kv, dh, dv, positions, window, keep, n_split, q.dtype, q.device)
    out = torch.empty(q.shape[0], round8(h * dv), dtype=q.dtype, device=q.device)
    sc = _lib.OharaMixedScores(scale, window, keep, 0, _ptr(temp), _ptr(talk))
    check(_typed("attn_mixed", q.dtype)(
        _ptr(q), _ptr(kcache), _ptr(vcache), h, h_kv, dh, dv, t_max, C.byref(sc), positions, n_split, _ptr(workspace), workspace.numel(),
        _ptr(out), out.stride(0), seq.ref, _stream()), "attn_mixed")
    return out


def latent_front(p, q_rank, off_c, rank, qn, cn, eps, cache, seq: Seq, compact: bool = False):
    """p rows [query latent; cached latent at off_c] -> RMS-normed query latent (rows, round8(q_rank)) and, with ``compact``, the
    normed cached latent (rows, round8(rank)), which goes into the cache (cache rows, positions, round8(rank)) either way."""
    q = torch.empty(p.shape[0], round8(q_rank), dtype=p.dtype, device=p.device)
    c = torch.empty(p.shape[0], round8(rank), dtype=p.dtype, device=p.device) if compact else None
    check(_typed("latent_front", p.dtype)(
        _ptr(p), p.stride(0), q_rank, off_c, rank, _ptr(qn), _ptr(cn), eps, _ptr(q), _ptr(cache), cache.shape[1], _ptr(c), seq.ref,
        _stream()), "latent_front")
    return q, c


def latent_rotary_front(p, h: int, dq: int, cos, sin, qr, head_stride: int, seq: Seq, *, cache=None, off_c=0, off_r=0, rank=0, cn=None,
                        eps=0.0, compact: bool = False):
    """p rows [h heads of dq unrotated and round8(rot) rotated elements; a latent at off_c; a rotated key part at off_r], see
    ohara_latent_rotary_front_*: the queries' rotated parts go to ``qr`` (rows, heads ``head_stride`` apart; may be a view of p), latent and
    key part, with ``cn``, into the cache and, ``compact``, into the returned (rows, round8(rank) + round8(rot))."""
    rot = 2 * cos.shape[1]
    if cos.shape != sin.shape or (cache is not None and (cache.shape[2] != round8(rank) + round8(rot) or cos.shape[0] < cache.shape[1])):
        raise ValueError("rotary tables and cache do not fit")
    t_max = cos.shape[0] if cache is None else cache.shape[1]
    c = torch.empty(p.shape[0], cache.shape[2], dtype=p.dtype, device=p.device) if compact else None
    check(_typed("latent_rotary_front", p.dtype)(
        _ptr(p), p.stride(0), h, dq, rot, _ptr(cos), _ptr(sin), _ptr(qr), qr.stride(0), head_stride, off_c, off_r, rank, _ptr(cn), eps,
        _ptr(cache), t_max, _ptr(c), seq.ref, _stream()), "latent_rotary_front")
    return c


def head_linear(x, w, n_out: int, gate=None, out=None, x_heads: int = 0, out_heads: int = 0):
    """x (rows, >= h * k), w (h, n, k) -> (rows, round8(h * n_out)): one matrix per head, the first n_out entries of each, times
    sigmoid(gate) with gate a (rows, h * n_out) column slice.  ``x_heads``, ``out_heads``: elements between neighbouring heads where
    they do not follow each other (``out`` is then the caller's)."""
    h, n, k = w.shape
    if out is None:
        out = torch.empty(x.shape[0], round8(h * n_out), dtype=x.dtype, device=x.device)
    check(_typed("head_linear", x.dtype)(
        _ptr(x), x.stride(0), _ptr(w), h, n, k, n_out, x.shape[0], _ptr(gate), 0 if gate is None else gate.stride(0), _ptr(out),
        out.stride(0), x_heads, out_heads, _stream()), "head_linear")
    return out


def attn_latent_workspace(rows, h, rank, n_split, device) -> torch.Tensor:
    n = lib().ohara_attn_latent_workspace_bytes(rows, h, rank, n_split)
    if n < 0:
        raise ValueError("bad latent attention workspace shape")
    return torch.empty(n, dtype=torch.uint8, device=device)


def attn_latent(q, cache, h, rank, scale, seq: Seq, n_split=1, workspace=None, window: int = 0):
    """q (rows, h * round8(rank)) against the cached latents (cache rows, positions, round8(rank)), which are keys and values at
    once -> weighted sums (rows, h * round8(rank)).  Rows of q and of the cache may be longer: what follows takes part in the scores only.
    ``window``: as in ``attn_scored``."""
    d_key = cache.shape[2] - round8(rank)
    if q.shape[1] != h * cache.shape[2]:
        raise ValueError("queries and cached rows differ in length")
    out = torch.empty(q.shape[0], h * round8(rank), dtype=q.dtype, device=q.device)
    check(_typed("attn_latent", q.dtype)(_ptr(q), _ptr(cache), h, rank, d_key, cache.shape[1], scale, window, n_split, _ptr(workspace), _ptr(out),
                                         seq.ref, _stream()), "attn_latent")
    return out


def delta_step(d: "_lib.OharaDelta", p, state, ring, seq: Seq):
    """One token per sequence of the gated delta rule -> (rows, round8(heads * vdim)); state and ring updated."""
    out = torch.empty(p.shape[0], round8(d.heads * d.vdim), dtype=p.dtype, device=p.device)
    check(_typed("delta_step", p.dtype)(C.byref(d), _ptr(p), p.stride(0), _ptr(state), _ptr(ring), _ptr(out), out.stride(0),
                                        seq.ref, _stream()), "delta_step")
    return out


def delta_workspace_bytes(heads, dim, vdim, batch, tokens) -> int:
    n = lib().ohara_delta_workspace_bytes(heads, dim, vdim, batch, tokens)
    if n < 0:
        raise ValueError("bad delta rule shape")
    return n


def delta_prefill(d: "_lib.OharaDelta", p, za, zg, state, ring, workspace, seq: Seq):
    """Any number of tokens per sequence of the gated delta rule (za, zg: the low-rank products, None where d has no such
    matrix); the ring is updated after the call's convolutions."""
    rows = p.shape[0]
    out = torch.empty(rows, round8(d.heads * d.vdim), dtype=p.dtype, device=p.device)
    o_tmp = torch.empty(rows, d.heads * d.vdim, dtype=F32, device=p.device)
    check(_typed("delta_prefill", p.dtype)(
        C.byref(d), _ptr(p), p.stride(0), _ptr(za), 0 if za is None else za.stride(0), _ptr(zg), 0 if zg is None else zg.stride(0),
        _ptr(state), _ptr(ring), _ptr(workspace), workspace.numel(), _ptr(o_tmp), _ptr(out), out.stride(0), seq.ref, _stream()), "delta_prefill")
    conv_ring_store(p, 2 * d.kv_heads * d.dim + d.heads * d.vdim, ring, seq)
    return out


def gemm_glu(x, w, limit: float, alpha: float, offset: float, out=None):
    """g sigmoid(alpha g) (u + offset), g = min(x Wg^T, limit), u = clamp(x Wu^T, +-limit); w: packed (bf16) or a pair of (n, k) fp32."""
    f32 = x.dtype == F32
    n, k = w[0].shape if f32 else (w.n, w.k)
    if not x.is_cuda or x.stride(1) != 1 or x.shape[1] != k:
        raise ValueError("x must be a device matrix with unit column stride and W's columns")
    if out is None:
        out = torch.empty(x.shape[0], n, dtype=x.dtype, device=x.device)
    ptrs = (_ptr(w[0]), _ptr(w[1])) if f32 else (_ptr(w.data),)
    check(_typed("gemm_glu", x.dtype)(_ptr(x), x.stride(0), *ptrs, n, k, limit, alpha, offset, x.shape[0], _ptr(out), out.stride(0),
                                      _stream()), "gemm_glu")
    return out


def moe_router(x, w, correction, k: int, top: int, groups: int, keep: int, counter, flags: int = 0):
    """x (rows, k), w (outputs, k) -> (idx (rows, top) int32, weights (rows, top) fp32, offs, pair_of, pos_of): see
    ohara_moe_router_*.  counter: one int32, zero between calls."""
    rows, n = x.shape[0], w.shape[0]
    i32 = lambda *s: torch.empty(*s, dtype=torch.int32, device=x.device)  # noqa: E731
    idx, wgt = i32(rows, top), torch.empty(rows, top, dtype=F32, device=x.device)
    offs, pair_of, pos_of, hist = i32(n + 1), i32(rows * top), i32(rows * top), i32((rows * top + 1023) // 1024 * n)
    check(_typed("moe_router", x.dtype)(
        _ptr(x), x.stride(0), _ptr(w), w.stride(0), _ptr(correction), rows, k, n, top, groups, keep, flags, _ptr(idx), _ptr(wgt), _ptr(offs),
        _ptr(pair_of), _ptr(pos_of), _ptr(hist), _ptr(counter), _stream()), "moe_router")
    return idx, wgt, offs, pair_of, pos_of


def retention_workspace_bytes(heads, dim, vdim, batch, tokens) -> int:
    n = lib().ohara_retention_workspace_bytes(heads, dim, vdim, batch, tokens)
    if n < 0:
        raise ValueError("bad retention shape")
    return n


def retention(r: "_lib.OharaRetention", p, state, workspace, seq: Seq, out=None):
    """Normed and gated heads (rows, heads * vdim) of the tokens in p; the state moves on.  One token per sequence needs no
    workspace.  ``out``: a column slice of a wider buffer."""
    n = r.heads * r.vdim
    if out is None:
        out = torch.empty(p.shape[0], n, dtype=p.dtype, device=p.device)
    elif out.shape != (p.shape[0], n) or out.dtype != p.dtype or out.stride(1) != 1:
        raise ValueError("out must be (rows, heads * vdim) with unit column stride")
    if seq.seq_len == 1:
        check(_typed("retention_step", p.dtype)(C.byref(r), _ptr(p), p.stride(0), _ptr(state), _ptr(out), out.stride(0), seq.ref, _stream()),
              "retention_step")
    else:
        check(_typed("retention_prefill", p.dtype)(C.byref(r), _ptr(p), p.stride(0), _ptr(state), _ptr(workspace), workspace.numel(),
                                                   _ptr(out), out.stride(0), seq.ref, _stream()), "retention_prefill")
    return out
