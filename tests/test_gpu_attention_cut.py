"""Decode attention whose context is cut by its own length: the lengths and numbers of (row, head) pairs where the cut changes, every
room for chunks, one position and one per sequence, against 64 bits and against the walk in one piece."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
LENGTHS = [1, 63, 320, 321, 384, 385, 641, 768, 769, 1100]


def _exact(q, k, v, lengths):
    """Bound: weights and result rounded to bf16 (2^-8 each), scores from fp32 sums that are 16 together at most."""
    B, H, D = q.shape
    want, bound = torch.empty(2, B, H, D, dtype=torch.float64, device=q.device)
    for b, L in enumerate(lengths):
        kk, vv = (t[b, :L].double().repeat_interleave(H // t.shape[2], 1).transpose(0, 1).contiguous() for t in (k, v))
        p = torch.softmax((kk @ q[b].double()[:, :, None]).squeeze(-1) / D ** 0.5, -1)[:, None]
        want[b] = (p @ vv).squeeze(1)
        bound[b] = want[b].abs() * 2.0 ** -8 + (p @ vv.abs()).squeeze(1) * (2.0 ** -8 + D * 2.0 ** -20)
    return want, bound + 1e-30


# (batch, heads, key heads): up to 80 pairs, up to 128, more
@pytest.mark.parametrize("B,H,Hkv", [(1, 4, 1), (16, 16, 4), (10, 16, 8), (9, 9, 9), (16, 8, 8), (43, 3, 3), (40, 16, 4)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("int8", [False, True])
def test_lengths_where_the_cut_changes(cuda, B, H, Hkv, D, int8):
    from ohara_amd import ops
    from ohara_amd.llama import KVCache

    T = max(LENGTHS) + 3
    g = torch.Generator(device=cuda).manual_seed(B + H + D)
    q = torch.randn(B, H * D, generator=g, device=cuda).to(BF)
    k, v = (torch.randn(B, T, Hkv, D, generator=g, device=cuda).to(BF) for _ in range(2))
    if int8:
        cache = KVCache((B, T, Hkv, D), T, 0, device=cuda, dtype=BF, int8=True)
        ops.kv_quant_append(k, v, cache, 0)

        def run(pos, ns, ws, seq_pos=None):
            return ops.attn_cached_int8(q, cache, H, Hkv, D, pos, ns, ws, seq_pos=seq_pos)
    else:
        def run(pos, ns, ws, seq_pos=None):
            return ops.attn_cached(q, k, v, H, Hkv, D, pos, ns, ws, seq_pos=seq_pos)
    whole = {}
    for L in LENGTHS:
        whole[L] = run(L - 1, 1, ops.attn_workspace(B, H, Hkv, D, 1, cuda))
        if not int8:
            want, bound = _exact(q.view(B, H, D), k, v, [L] * B)
            assert ((whole[L].view(B, H, D).double() - want).abs() <= bound).all()
    rooms = {ns: ops.attn_workspace(B, H, Hkv, D, ns, cuda) for ns in (2, 3, 7, 16, 33)}
    for L in LENGTHS:  # one workspace for every length: its counters have to come back to zero
        scale = whole[L].float().abs().max().item()
        for ns, ws in rooms.items():
            # another order of fp32 sums: at most the last bf16 place at the output's scale
            assert (run(L - 1, ns, ws).float() - whole[L].float()).abs().max().item() <= scale * 2.0 ** -8
    # every sequence at its own position: each is cut by its own length
    lengths = [LENGTHS[b % len(LENGTHS)] for b in range(B)]
    pos = torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device=cuda)
    for ns, ws in rooms.items():
        got = run(0, ns, ws, seq_pos=pos)
        for b, L in enumerate(lengths):
            scale = whole[L][b].float().abs().max().item()
            assert (got[b].float() - whole[L][b].float()).abs().max().item() <= scale * 2.0 ** -8


@pytest.mark.parametrize("B,H,Hkv,D", [(16, 8, 8, 128), (12, 32, 8, 128), (12, 8, 8, 64)])
def test_lengths_around_4096(cuda, B, H, Hkv, D):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(B + H + D)
    q = torch.randn(B, H * D, generator=g, device=cuda).to(BF)
    k, v = (torch.randn(B, 4200, Hkv, D, generator=g, device=cuda).to(BF) for _ in range(2))
    rooms = {ns: ops.attn_workspace(B, H, Hkv, D, ns, cuda) for ns in (8, 10, 33)}
    for L in (4096, 4097, 4161):
        want, bound = _exact(q.view(B, H, D), k, v, [L] * B)
        for ns, ws in rooms.items():
            got = ops.attn_cached(q, k, v, H, Hkv, D, L - 1, ns, ws)
            assert ((got.view(B, H, D).double() - want).abs() <= bound).all()


# a number of pairs of every kind of line (one workgroup a CU, two, all there is room for), the room that callers ask for
@pytest.mark.parametrize("B,H,Hkv", [(4, 24, 6), (6, 8, 8), (9, 16, 8), (25, 4, 4), (25, 32, 8), (50, 6, 6)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("int8", [False, True])
def test_longer_contexts(cuda, B, H, Hkv, D, int8):
    from ohara_amd import ops
    from ohara_amd.llama import KVCache

    T, ns = 3300, 1024 // (B * Hkv)
    g = torch.Generator(device=cuda).manual_seed(B + H + D)
    q = torch.randn(B, H * D, generator=g, device=cuda).to(BF)
    k, v = (torch.randn(B, T, Hkv, D, generator=g, device=cuda).to(BF) for _ in range(2))
    ws, one = (ops.attn_workspace(B, H, Hkv, D, n, cuda) for n in (ns, 1))
    if int8:
        cache = KVCache((B, T, Hkv, D), T, 0, device=cuda, dtype=BF, int8=True)
        ops.kv_quant_append(k, v, cache, 0)
    for L in (321, 449, 640, 1025, 1536, 3201):
        if int8:
            got, whole = (ops.attn_cached_int8(q, cache, H, Hkv, D, L - 1, n, w).float() for n, w in ((ns, ws), (1, one)))
            # another order of fp32 sums: a value may round to its neighbour, 2^-7 of it at most
            assert ((got - whole).abs() <= whole.abs() * 2.0 ** -7 + 2.0 ** -16).all()
        else:
            want, bound = _exact(q.view(B, H, D), k, v, [L] * B)
            assert ((ops.attn_cached(q, k, v, H, Hkv, D, L - 1, ns, ws).view(B, H, D).double() - want).abs() <= bound).all()
