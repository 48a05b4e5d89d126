"""The tiles whose waves work in two halves, those that fill the chip once with few rows, and the rotary epilogue by whole rows of the tables:
depths that end inside a step, with one and before the ring is full, against the same rows in calls of 32 that run small tiles, bit for bit, and against 64 bits; rotated rows
against the plain product's, rotated here."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

# tile, rows, packed rows, K: one step, a step and a piece, less than the ring, every remainder of 64 that counts (8, 32, 40, 0)
CASES = [
    (128192, 1025, 4112, 64), (128192, 1025, 4112, 72), (128192, 1025, 4112, 128), (128192, 1025, 4112, 168), (128192, 1100, 4112, 264),
    (128192, 1024, 6144, 776), (128256, 3000, 2320, 328), (128256, 2049, 3088, 520), (128256, 1537, 4112, 544), (128256, 2049, 3088, 768),
    (256256, 3000, 8208, 168), (256256, 3000, 8208, 192), (256256, 3000, 8208, 200), (256256, 2049, 6160, 296), (256256, 2049, 6160, 320),
    (256256, 1537, 8208, 360),
    (64048, 128, 6128, 520), (64048, 190, 3056, 776), (64048, 65, 6128, 544), (64096, 100, 11280, 1032), (64096, 500, 3056, 1096), (64096, 470, 3056, 1024),
]


@pytest.mark.parametrize("tile,rows,packed,k", CASES)
def test_tiles_and_small_ones(cuda, tile, rows, packed, k):
    from ohara_amd import ops
    from ohara_amd._lib import lib

    assert lib().ohara_gemm_tile_of(rows, packed, k) == tile
    g = torch.Generator(device=cuda).manual_seed(rows + packed + k)
    x = (torch.randn(rows, k, generator=g, device=cuda) * 3).to(BF)
    w = (torch.randn(packed, k, generator=g, device=cuda) * 0.3).to(BF)
    w[5, k - 1] = float("inf")  # (past K the walk stands in other values: none of them may be multiplied, not even by zero)
    x[:, k - 1] = x[:, k - 1].abs() + 1
    spans = [slice(r, min(r + 32, rows)) for r in range(0, rows, 32)]
    wp, res = ops.pack_linear(w), torch.randn(rows, packed, generator=g, device=cuda).to(BF)
    got, summed = ops.gemm(x, wp), ops.gemm(x, wp, residual=res)
    assert torch.equal(got, torch.cat([ops.gemm(x[s], wp) for s in spans]))
    assert torch.equal(summed, torch.cat([ops.gemm(x[s], wp, residual=res[s]) for s in spans]))
    assert (got[:, 5] == float("inf")).all()
    for f in (packed // 2, packed // 2 - 3):
        gates = ops.pack_gate_up(w[:f].contiguous(), w[f:2 * f].contiguous())
        assert torch.equal(ops.gemm(x, gates), torch.cat([ops.gemm(x[s], gates) for s in spans]))
    cols = torch.cat([torch.arange(5), torch.arange(6, packed)])
    xd, wd = x.double(), w[cols.to(cuda)].double()
    want = xd @ wd.t()
    # one rounding to bf16 of the result and K roundings to fp32 of partial sums
    bound = want.abs() * 2.0 ** -8 + k * 2.0 ** -24 * (xd.abs() @ wd.abs().t()) + 1e-30
    assert ((got[:, cols.to(cuda)].double() - want).abs() <= bound).all()


# head width, query heads, key heads, sequences, positions of each, K: strips two and four a wave, heads narrower than a wave's strips,
# sequences that end inside a tile, all tiles from 64 rows on
ROTARY = [
    (128, 6, 6, 2, 1024, 136), (128, 16, 4, 1, 2049, 200), (128, 6, 6, 8, 1024, 64), (64, 16, 16, 3, 700, 192), (64, 32, 8, 1, 3000, 520), (32, 40, 2, 2, 600, 72),
    (128, 6, 6, 1, 400, 768), (64, 5, 5, 1, 97, 136), (48, 10, 2, 2, 777, 96), (16, 60, 4, 1, 1500, 72),
]


@pytest.mark.parametrize("D,H,Hkv,B,S,k", ROTARY)
def test_rotary_by_rows_of_the_tables(cuda, D, H, Hkv, B, S, k):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(D + H + S)
    pos, T = 5, S + 9
    x = torch.randn(B, S, k, generator=g, device=cuda).to(BF)
    w = (torch.randn((H + 2 * Hkv) * D, k, generator=g, device=cuda) * 0.1).to(BF)
    ang = torch.rand(T, D // 2, generator=g, device=cuda) * 6.28
    cos, sin = ang.cos().to(BF), ang.sin().to(BF)
    wq = ops.pack_qkv(w[:H * D], w[H * D:(H + Hkv) * D], w[(H + Hkv) * D:])
    keys, values = (torch.full((B, T, Hkv, D), 9.0, dtype=BF, device=cuda) for _ in range(2))
    q = ops.qkv_rope_append(x.view(B * S, k), wq, None, 1e-5, H, Hkv, D, cos, sin, pos, keys, values, seq_len=S).view(B, S, H, D)
    y = ops.gemm(x.view(B * S, k), ops.pack_linear(w)).view(B, S, H + 2 * Hkv, D)  # rounded, as the rotation takes it
    e, o = y[..., 0::2].float(), y[..., 1::2].float()
    c, n = (t[pos:pos + S].float().view(1, S, 1, D // 2) for t in (cos, sin))
    turned = torch.stack([e * c - o * n, e * n + o * c], -1).flatten(-2).to(BF)
    assert torch.equal(q, turned[:, :, :H]) and torch.equal(keys[:, pos:pos + S], turned[:, :, H:H + Hkv])
    assert torch.equal(values[:, pos:pos + S], y[:, :, H + Hkv:])
    for cache in (keys, values):
        assert (cache[:, :pos] == 9.0).all() and (cache[:, pos + S:] == 9.0).all()
