"""The tiled GEMM over its six tiles: edges of tiles, ragged rows, strips and K, row strides and row starts of any alignment,
against the product of the same bf16 values in 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _bound(x, w, y):
    """One rounding to bf16 of the result and K roundings to fp32 of partial sums."""
    return y.abs() * 2.0 ** -8 + x.shape[1] * 2.0 ** -24 * (x.abs() @ w.abs().t()) + 1e-30


# (rows, columns, K): the comment names the tile that the rule picks
SHAPES = [
    (65, 16, 8), (97, 40, 72), (320, 768, 768), (129, 1000, 520), (257, 2048, 2056),  # 32 x 32; K below, at and past a step
    (96, 6144, 768), (700, 1504, 1000), (193, 4100, 768),                             # 64 x 64
    (320, 6144, 712),                                                                 # 64 x 128
    (1000, 3096, 2008), (1030, 6104, 264),                                            # 128 x 128
    (2049, 2304, 768), (700, 6160, 776), (2100, 11264, 520),                          # 128 x 192
    (700, 17928, 1032),                                                               # 256 x 256
]


@pytest.mark.parametrize("rows,n,k", SHAPES)
def test_tiles_and_their_edges(cuda, rows, n, k):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(rows * 31 + n * 7 + k)
    x = torch.randn(rows, k, generator=g, device=cuda).to(BF)
    w = (torch.randn(n, k, generator=g, device=cuda) * 0.05).to(BF)
    res = torch.randn(rows, n, generator=g, device=cuda).to(BF)
    xd, wd = x.double(), w.double()
    want = xd @ wd.t()
    packed = ops.pack_linear(w)
    got = ops.gemm(x, packed)
    assert ((got.double() - want).abs() <= _bound(xd, wd, want)).all()
    summed = ops.gemm(x, packed, residual=res)
    assert torch.equal(summed, (res.float() + got.float()).to(BF))  # the sum of the two rounded values, rounded once


@pytest.mark.parametrize("rows,n,k", [(70, 48, 24), (200, 768, 136), (900, 3072, 768)])
@pytest.mark.parametrize("start,stride", [(0, 16), (1, 0), (3, 8), (8, 24)])
def test_rows_that_start_anywhere(cuda, rows, n, k, start, stride):
    """Rows apart by more than K, and starts that are not on 16 bytes (they take the loads through registers)."""
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(5)
    flat = torch.randn(rows * (k + stride) + 16, generator=g, device=cuda).to(BF)
    x = torch.as_strided(flat, (rows, k), (k + stride, 1), start)
    w = (torch.randn(n, k, generator=g, device=cuda) * 0.05).to(BF)
    assert torch.equal(ops.gemm(x, ops.pack_linear(w)), ops.gemm(x.contiguous(), ops.pack_linear(w)))


def test_infinities_stay_in_their_row(cuda):
    """What is multiplied by padding (columns past K, rows and strips past the end) never reaches a result."""
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(6)
    x = torch.randn(130, 72, generator=g, device=cuda).to(BF)
    w = torch.randn(40, 72, generator=g, device=cuda).to(BF)
    x[17, 64:] = float("inf")
    x[129, 3] = float("nan")
    got = ops.gemm(x, ops.pack_linear(w))
    fine = [r for r in range(130) if r not in (17, 129)]
    assert got[fine].isfinite().all() and got[129].isnan().all()
    want = x[17].double() @ w.double().t()
    assert torch.equal(got[17].isnan(), want.isnan())
    at = ~want.isnan()
    assert torch.equal(got[17][at].double(), want[at])


@pytest.mark.parametrize("rows,n,k", SHAPES)
def test_infinite_weights_of_a_last_step(cuda, rows, n, k):
    """An infinite weight in the last columns makes its own column of the result infinite and no NaN, also where K ends inside a step."""
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(7)
    x = torch.rand(rows, k, generator=g, device=cuda).add_(0.5).to(BF)
    w = torch.randn(n, k, generator=g, device=cuda).to(BF)
    w[3, k - 1], w[n - 2, k - 8] = float("inf"), -float("inf")
    got = ops.gemm(x, ops.pack_linear(w))
    assert (got[:, 3] == float("inf")).all() and (got[:, n - 2] == -float("inf")).all()
    rest = [c for c in range(n) if c not in (3, n - 2)]
    assert got[:, rest].isfinite().all()


# 96 rows take tiles that are 32 rows high, 4100 tiles of 192 columns, 9000 tiles of 256
@pytest.mark.parametrize("rows,f", [(96, 264), (300, 3072), (1100, 1544), (2100, 5632), (4100, 1160), (9000, 3080)])
@pytest.mark.parametrize("pad", [0, 1, 4])
def test_stores_of_16_bytes_and_less(cuda, rows, f, pad):
    """Gates and sums stored 16 bytes a lane, and through rows that leave no room for that: the same bits; and the gates of the skinny
    kernels, which have their reciprocal from another unit."""
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(rows + f)
    k = 72
    x = (torch.randn(rows, k, generator=g, device=cuda) * 4).to(BF)
    wg, wu = ((torch.randn(f, k, generator=g, device=cuda)).to(BF) for _ in range(2))
    gates, flat = ops.pack_gate_up(wg, wu), ops.pack_linear(wg)
    odd = torch.full((rows, f + pad), 7.0, dtype=BF, device=cuda)
    ops.gemm(x, gates, out=odd[:, :f])
    skinny = torch.cat([ops.gemm_skinny(x[i:i + 64], gates) for i in range(0, min(rows, 320), 64)])[:320]
    assert (odd[:320, :f] != skinny).float().mean() <= 0.01  # sums over K in another order: last places
    gate, up = (x.double() @ w.double().t() for w in (wg, wu))
    want = gate * torch.sigmoid(gate) * up
    # silu, up and product are each rounded to bf16, and the gate, which silu follows with a slope of at most 1.1; sums are in fp32
    err_gate, err_up = (k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) for w in (wg, wu))
    silu = (gate * torch.sigmoid(gate)).abs()
    bound = 1.02 * (silu * (up.abs() * 3 * 2.0 ** -8 + err_up) + 1.1 * (gate.abs() * 2.0 ** -8 + err_gate) * up.abs()) + 1e-30
    assert ((odd[:, :f].double() - want).abs() <= bound).all()
    assert (odd[:, f:] == 7.0).all()
    res = torch.randn(rows, f + pad, generator=g, device=cuda).to(BF)
    for resid in (None, res[:, :f]):
        ops.gemm(x, flat, residual=resid, out=odd[:, :f])
        assert torch.equal(odd[:, :f], ops.gemm(x, flat, residual=None if resid is None else resid.contiguous()))
        assert (odd[:, f:] == 7.0).all()


def test_gate_of_every_value(cuda):
    """silu over every bf16 number, the ones where its short form does not hold among them, against the kernel of few rows."""
    from ohara_amd import ops

    v = torch.arange(-32768, 32768, dtype=torch.int32, device=cuda).to(torch.int16).view(BF)
    v = v[v.isfinite()]
    v = torch.cat([v, torch.zeros(-v.numel() % 64, dtype=BF, device=cuda)])
    v = v.view(64, -1).t().contiguous().view(-1)  # rows of a fragment from all over the range
    x = torch.zeros(v.numel(), 8, dtype=BF, device=cuda)
    x[:, 0], x[:, 1] = v, 1.0
    wg, wu = (torch.zeros(64, 8, dtype=BF, device=cuda) for _ in range(2))
    wg[:, 0], wu[:, 1] = 1.0, 1.0
    w = ops.pack_gate_up(wg, wu)
    for part in (x, x[x[:, 0] > -87]):  # the second without a row that takes the long form
        got = ops.gemm(part, w)
        want = torch.cat([ops.gemm_skinny(part[i:i + 64].contiguous(), w) for i in range(0, part.shape[0], 64)])
        assert torch.equal(got, want)


@pytest.mark.parametrize("B,S,H,Hkv,D,K", [(2, 100, 6, 6, 128, 768), (3, 90, 3, 1, 48, 64), (5, 300, 5, 5, 80, 136), (1, 2100, 9, 3, 64, 328),
                                           (9, 1000, 16, 4, 128, 520)])
def test_rotary_regions_and_their_edges(cuda, B, S, H, Hkv, D, K):
    """Strips of q, k and v side by side in one store, also where the regions start on an odd strip, against 64 bits."""
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(S)
    pos, T = 3, S + 8
    x = torch.randn(B * S, K, generator=g, device=cuda).to(BF)
    wq, wk, wv = ((torch.randn(n * D, K, generator=g, device=cuda) * 0.1).to(BF) for n in (H, Hkv, Hkv))
    ang = torch.rand(T, D // 2, generator=g, device=cuda) * 6.28
    cos, sin = ang.cos().to(BF), ang.sin().to(BF)
    kc, vc = (torch.full((B, T, Hkv, D), 9.0, dtype=BF, device=cuda) for _ in range(2))
    q = ops.qkv_rope_append(x, ops.pack_qkv(wq, wk, wv), None, 1e-5, H, Hkv, D, cos, sin, pos, kc, vc, seq_len=S).view(B, S, H, D)
    assert (kc[:, :pos] == 9.0).all() and (kc[:, pos + S:] == 9.0).all()
    assert (vc[:, :pos] == 9.0).all() and (vc[:, pos + S:] == 9.0).all()

    def plain(w, n):
        y, mass = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
        return y.view(B, S, n, D), (y.abs() * 2.0 ** -8 + K * 2.0 ** -24 * mass).view(B, S, n, D)

    def turned(w, n):
        y, e = plain(w, n)
        c, s = (t[pos:pos + S].double()[None, :, None] for t in (cos, sin))
        a, b, ea, eb = y[..., 0::2], y[..., 1::2], e[..., 0::2], e[..., 1::2]
        want = torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)
        bound = torch.stack([ea * c.abs() + eb * s.abs(), ea * s.abs() + eb * c.abs()], -1).flatten(-2)
        return want, bound + want.abs() * 2.0 ** -8 + bound * 2.0 ** -7

    for got, (want, bound) in ((q, turned(wq, H)), (kc[:, pos:pos + S], turned(wk, Hkv)), (vc[:, pos:pos + S], plain(wv, Hkv))):
        assert ((got.double() - want).abs() <= bound + 1e-30).all()
