"""Attention over many query positions in its four workgroup shapes: tile edges, queries and positions that do not fill them, heads that divide over the XCDs and heads that do not, caches that start on any element."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _reference(q, k, v, pos):
    """In 64 bits, with the bound: weights are rounded to bf16 (2^-8 of each, all of a query's in one direction at worst, against
    a sum of unrounded ones), the result once more; a score is an fp32 sum of D products that are 16 together at most, which its
    weight follows."""
    B, S, H, D = q.shape
    L = pos + S
    k = k[:, :L].double().repeat_interleave(H // k.shape[2], 2)
    v = v[:, :L].double().repeat_interleave(H // v.shape[2], 2)
    s = torch.matmul(q.double().transpose(1, 2), k.permute(0, 2, 3, 1).contiguous()) / D ** 0.5
    s.masked_fill_(torch.arange(L, device=q.device)[None, :] > pos + torch.arange(S, device=q.device)[:, None], float("-inf"))
    p = torch.softmax(s, -1)
    vt = v.transpose(1, 2).contiguous()
    want = torch.matmul(p, vt).transpose(1, 2)
    mass = torch.matmul(p, vt.abs()).transpose(1, 2)
    return want, want.abs() * 2.0 ** -8 + mass * (2.0 ** -8 + D * 2.0 ** -20) + 1e-30


# (batch, queries, heads, key heads, position before them): the comment names the workgroup that the rule picks at 128 columns
SHAPES = [
    (1, 16, 2, 1, 0), (1, 17, 6, 6, 15), (3, 33, 8, 2, 30), (4, 48, 16, 4, 1000), (1, 257, 8, 8, 31),   # a team of 16
    (1, 1000, 7, 7, 0), (2, 513, 6, 2, 63), (8, 32, 24, 8, 97),                                         # two teams
    (2, 1030, 12, 3, 1), (1, 577, 24, 24, 64), (8, 32, 24, 8, 96),                                      # waves of 16
    (3, 60, 300, 300, 10), (3, 129, 70, 70, 130), (3, 250, 70, 70, 249),                                # waves of 16
    (8, 520, 32, 4, 3), (3, 130, 131, 131, 63),                                                         # waves of 32
    (5, 65, 64, 8, 0), (3, 128, 86, 43, 5), (3, 250, 70, 70, 250), (2, 200, 170, 34, 9),                # waves of 32
]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,H,Hkv,pos", SHAPES)
def test_shapes_and_their_edges(cuda, B, S, H, Hkv, pos, D):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(B + S * 3 + H * 7 + pos)
    q = (torch.randn(B, S, H, D, generator=g, device=cuda) * 2).to(BF)
    k, v = (torch.randn(B, pos + S + 3, Hkv, D, generator=g, device=cuda).to(BF) for _ in range(2))
    want, bound = _reference(q, k, v, pos)
    k[:, pos + S:] = float("nan")  # what lies behind the fed tokens is never used
    v[:, pos + S:] = float("nan")
    got = ops.attn_prefill(q.view(B * S, H * D), k, v, H, Hkv, D, pos, S).view(B, S, H, D)
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,H,Hkv,pos", [(1, 40, 4, 2, 70), (2, 300, 6, 6, 5), (4, 200, 16, 4, 0)])
@pytest.mark.parametrize("start", [2, 4])
def test_caches_that_start_anywhere(cuda, B, S, H, Hkv, pos, D, start):
    """Caches that are not on 16 bytes take the loads through registers."""
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(S)
    shape = (B, pos + S, Hkv, D)
    n = B * (pos + S) * Hkv * D
    q = torch.randn(B, S, H, D, generator=g, device=cuda).to(BF)
    k, v = (torch.randn(n + 16, generator=g, device=cuda).to(BF)[start:start + n].view(shape) for _ in range(2))
    want, bound = _reference(q, k, v, pos)
    got = ops.attn_prefill(q.view(B * S, H * D), k, v, H, Hkv, D, pos, S).view(B, S, H, D)
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("B,S,H,pos", [(1, 256, 6, 100), (1, 700, 8, 0), (2, 900, 12, 7)])
def test_infinities_reach_no_query_before_their_tile(cuda, B, S, H, pos):
    """An infinite value at one position: what sees it is not finite, and every query whose walk ends before the position's tile
    of 64 does not depend on it."""
    from ohara_amd import ops

    D = 128
    g = torch.Generator(device=cuda).manual_seed(S)
    q, k, v = (torch.randn(B, n, H, D, generator=g, device=cuda).to(BF) for n in (S, pos + S, pos + S))
    at = pos + S // 2
    clean = ops.attn_prefill(q.view(B * S, H * D), k, v, H, H, D, pos, S).view(B, S, H, D)
    v[:, at] = float("inf")
    got = ops.attn_prefill(q.view(B * S, H * D), k, v, H, H, D, pos, S).view(B, S, H, D)
    first = max(0, at // 64 * 64 - 32 - pos)  # 32: queries of one wave
    assert torch.equal(got[:, :first], clean[:, :first])
    assert not got[:, at - pos:].isfinite().any()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,H,Hkv,pos", [
    (1, 16, 6, 6, 509), (1, 17, 16, 4, 700), (1, 1, 4, 4, 1500), (2, 100, 6, 6, 765), (1, 33, 12, 4, 1000),    # three tiles a chunk and more
    (1, 200, 16, 4, 1400), (8, 100, 6, 6, 1200), (1, 1100, 2, 1, 0), (3, 190, 1, 1, 3000),                    # chunks some queries do not see
    (1, 700, 3, 1, 129), (1, 250, 6, 2, 1030),
])
def test_chunks_of_a_long_context(cuda, B, S, H, Hkv, pos, D):
    """Few queries behind many positions are cut into chunks; without room for their partial results they are not."""
    from ohara_amd import ops
    from ohara_amd._lib import check, lib

    g = torch.Generator(device=cuda).manual_seed(B + S * 3 + H * 7 + pos)
    q = (torch.randn(B, S, H, D, generator=g, device=cuda) * 2).to(BF)
    k, v = (torch.randn(B, pos + S + 3, Hkv, D, generator=g, device=cuda).to(BF) for _ in range(2))
    want, bound = _reference(q, k, v, pos)
    k[:, pos + S:] = float("nan")
    v[:, pos + S:] = float("nan")
    room = lib().ohara_attn_prefill_ws_bytes(B, S, H, Hkv, D, pos)
    assert room > 0 and lib().ohara_attn_prefill_ws_bytes(B, S, H, Hkv, D, pos + 2000) >= room
    whole = torch.empty(B * S, H * D, dtype=BF, device=cuda)

    def run(at, size):
        check(lib().ohara_attn_prefill_ws_bf16(q.data_ptr(), k.data_ptr(), v.data_ptr(), B, S, H, Hkv, D, k.shape[1], pos,
                                               whole.data_ptr(), at, size, torch.cuda.current_stream().cuda_stream), "attn_prefill")
        return whole.view(B, S, H, D)

    ws = torch.full((room + 64,), 0xFF, dtype=torch.uint8, device=cuda)  # NaNs: what no chunk wrote is never used
    for got in (ops.attn_prefill(q.view(B * S, H * D), k, v, H, Hkv, D, pos, S).view(B, S, H, D), run(ws.data_ptr(), room)):
        assert ((got.double() - want).abs() <= bound).all()
    assert (ws[room:] == 0xFF).all()
    for at, size in ((None, 0), (None, room), (ws.data_ptr(), 16)):
        assert ((run(at, size).double() - want).abs() <= bound).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,H,Hkv,pos,wins", [
    (1, 2, 6, 6, 400, (0, 0)), (1, 2, 6, 6, 900, (1, 1)), (1, 15, 6, 6, 368, (0, 0)), (3, 7, 5, 5, 376, (0, 0)), (3, 7, 5, 5, 377, (1, 1)),
    (2, 8, 16, 16, 119, (0, 0)), (2, 8, 16, 16, 120, (0, 1)), (4, 8, 16, 16, 0, (1, 1)), (8, 9, 8, 4, 300, (0, 1)), (8, 9, 4, 2, 300, (0, 0)),
    (1, 2, 6, 2, 0, (1, 1)), (2, 5, 16, 4, 33, (1, 1)), (1, 3, 20, 4, 700, (1, 1)), (8, 15, 6, 6, 3000, (1, 1)),
])
def test_a_few_tokens_a_sequence(cuda, B, S, H, Hkv, pos, wins, D):
    """Either kernel within the bound on both sides of the lines between them (wins: with heads of 64, of 128), and the one that is taken."""
    from ohara_amd import ops
    from ohara_amd._lib import lib

    assert lib().ohara_attn_prefill_wins(B, S, H, Hkv, D, pos) == wins[D == 128]
    g = torch.Generator(device=cuda).manual_seed(B + S * 3 + H * 7 + pos)
    q = (torch.randn(B, S, H, D, generator=g, device=cuda) * 2).to(BF)
    k, v = (torch.randn(B, pos + S + 3, Hkv, D, generator=g, device=cuda).to(BF) for _ in range(2))
    want, bound = _reference(q, k, v, pos)
    rows = q.view(B * S, H * D)
    assert ((ops.attn_cached(rows, k, v, H, Hkv, D, pos, 1, None, None, None, S).view(B, S, H, D).double() - want).abs() <= bound).all()
    k[:, pos + S:] = float("nan")
    v[:, pos + S:] = float("nan")
    assert ((ops.attn_prefill(rows, k, v, H, Hkv, D, pos, S).view(B, S, H, D).double() - want).abs() <= bound).all()
    assert ((ops.attn_auto(rows, k, v, H, Hkv, D, pos, 1, None, S).view(B, S, H, D).double() - want).abs() <= bound).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("S,pos", [(16, 700), (40, 2500)])  # four chunks, and more than one round of eight
def test_an_infinite_value_in_the_last_chunk_stays_infinite(cuda, S, pos, D):
    """The merge reads the last chunk again where its round of eight has no more: those sums are not added, not even times zero."""
    from ohara_amd import ops
    from ohara_amd._lib import lib

    H = 6
    assert lib().ohara_attn_prefill_ws_bytes(1, S, H, H, D, pos) > 0
    g = torch.Generator(device=cuda).manual_seed(S + D)
    q, k, v = (torch.randn(1, n, H, D, generator=g, device=cuda).to(BF) for n in (S, pos + S, pos + S))
    want, bound = _reference(q, k, v, pos)
    v[:, pos - 1, :, 0] = float("inf")
    got = ops.attn_prefill(q.view(S, H * D), k, v, H, H, D, pos, S).view(1, S, H, D)
    assert (got[..., 0] == float("inf")).all()
    assert ((got.double() - want).abs() <= bound)[..., 1:].all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,H,Hkv,pos", [
    (1, 2, 6, 6, 900), (2, 15, 16, 4, 1000), (1, 9, 20, 4, 700), (1, 15, 6, 2, 570),  # chunks, the new tokens in one tile and across two
    (4, 8, 16, 16, 0), (2, 5, 16, 4, 33), (1, 15, 6, 2, 56),                         # a team of four waves
    (40, 3, 16, 16, 20), (20, 15, 32, 8, 60), (70, 2, 8, 8, 126),                    # waves
])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_a_few_tokens_do_not_see_values_behind_them(cuda, B, S, H, Hkv, pos, D, value):
    """Two to fifteen tokens a sequence: a value that is not finite reaches the tokens from its own on, in its own column, and no others."""
    from ohara_amd import ops
    from ohara_amd._lib import lib

    assert lib().ohara_attn_prefill_wins(B, S, H, Hkv, 128, pos)
    g = torch.Generator(device=cuda).manual_seed(B + S + H + pos)
    q, k, v = (torch.randn(B, n, h, D, generator=g, device=cuda).to(BF) for n, h in ((S, H), (pos + S, Hkv), (pos + S, Hkv)))
    want, bound = _reference(q, k, v, pos)
    odd = torch.empty(v.numel() + 2, dtype=BF, device=cuda)[2:].view(v.shape)  # (a cache that is not on 16 bytes)
    for cache in (v.clone(), odd):
        for at in {1, S // 2, S - 1}:
            cache.copy_(v)
            cache[:, pos + at, Hkv - 1, 5] = value
            got = ops.attn_prefill(q.view(B * S, H * D), k, cache, H, Hkv, D, pos, S).view(B, S, H, D)
            seen = (slice(None), slice(at, None), slice(H - H // Hkv, None), 5)
            assert got[seen].isnan().all() if value != value else (got[seen] == value).all()
            got[seen] = want[seen].to(BF)
            assert ((got.double() - want).abs() <= bound).all()
