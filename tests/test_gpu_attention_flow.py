"""Attention whose softmax runs a tile behind its products: the same bits as in calls of sixteen queries, which four waves share, from walks
of three tiles on, ends inside a tile and with one, positions before them of any number, heads over the XCDs and not; infinities stay in the queries that see them."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

# batch, queries, heads, key heads, positions before them: more than 256 workgroups of 32 queries (512 of 16 with heads of 64), fewer than 768 of 128
SHAPES = [
    (1, 192, 90, 90, 0), (1, 193, 88, 8, 0), (2, 256, 40, 8, 0), (1, 257, 72, 72, 0), (1, 320, 60, 20, 2), (1, 450, 42, 6, 37), (2, 129, 120, 120, 63),
    (2, 448, 24, 24, 64), (3, 130, 80, 40, 65), (4, 66, 100, 100, 127), (1, 500, 48, 16, 12), (2, 250, 48, 48, 133),
]


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,S,H,Hkv,pos", SHAPES)
@pytest.mark.parametrize("odd", [None, "key", "value"])
def test_the_bits_of_calls_of_sixteen(cuda, B, S, H, Hkv, pos, D, odd):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(B + S * 3 + H * 7 + pos)
    q = (torch.randn(B, S, H, D, generator=g, device=cuda) * 2).to(BF)
    k, v = (torch.randn(B, pos + S + 3, Hkv, D, generator=g, device=cuda).to(BF) for _ in range(2))
    if odd:  # at the first positions of tiles (a masked value of a tile that a query walks weighs zero, and makes an infinity a NaN;
        # no call of sixteen ends with one, whose copies stand in for what lies behind)
        (k if odd == "key" else v)[:, 64, :, 3] = float("inf")
        (k if odd == "key" else v)[:, (pos + S - 1) // 64 * 64, :, 5] = float("-inf")
    k[:, pos + S:] = float("nan")
    v[:, pos + S:] = float("nan")
    got = ops.attn_prefill(q.view(B * S, H * D), k, v, H, Hkv, D, pos, S).view(B, S, H * D)
    for b in range(B):
        for s in range(0, S - 31, 16):  # the last call takes what is left, 16 to 31 queries
            n = 16 if s + 32 <= S - 16 else S - s
            want = ops.attn_prefill(q[b, s:s + n].reshape(n, H * D), k[b:b + 1], v[b:b + 1], H, Hkv, D, pos + s, n)
            assert torch.allclose(got[b, s:s + n], want, rtol=0, atol=0, equal_nan=True)
    if not odd:
        assert torch.isfinite(got).all()


# batch, queries, heads, key heads, head width, positions before them: 32 queries a wave, a tile that begins or ends between a wave's sixteens among them
WIDE = [(32, 70, 24, 24, 64, 37), (28, 100, 24, 8, 64, 16), (22, 65, 24, 24, 128, 37), (17, 128, 32, 8, 128, 48), (24, 97, 16, 16, 128, 0), (9, 300, 32, 8, 128, 21),
        (13, 200, 32, 32, 64, 5)]


@pytest.mark.parametrize("B,S,H,Hkv,D,pos", WIDE)
def test_the_bits_of_32_queries_a_wave(cuda, B, S, H, Hkv, D, pos):
    """Wherever the queries stand: a sixteen whose tile needs no mask is scaled as where it has a wave to itself."""
    from ohara_amd import ops

    wide, halves = (-(-S // n) * H * B for n in (128, 64))
    assert 2 * halves >= 3 * wide and (wide >= 768 or (halves > 1280 if D == 64 else wide > 256 and S <= 128))
    g = torch.Generator(device=cuda).manual_seed(B + S)
    q = (torch.randn(B, S, H, D, generator=g, device=cuda) * 2).to(BF)
    k, v = (torch.randn(B, pos + S, Hkv, D, generator=g, device=cuda).to(BF) for _ in range(2))
    got = ops.attn_prefill(q.view(B * S, H * D), k, v, H, Hkv, D, pos, S).view(B, S, H * D)
    for b in (0, B - 1):
        for s in range(0, S - 31, 16):
            n = 16 if s + 32 <= S - 16 else S - s
            want = ops.attn_prefill(q[b, s:s + n].reshape(n, H * D), k[b:b + 1], v[b:b + 1], H, Hkv, D, pos + s, n)
            assert torch.equal(got[b, s:s + n], want)
