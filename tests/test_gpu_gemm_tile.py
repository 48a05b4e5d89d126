"""The tiled GEMM over its six tiles: edges of tiles, ragged rows, strips and K, row strides and row starts of any alignment,
against the product of the same bf16 values in 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _bound(x, w, y):
    """One rounding to bf16 of the result and K roundings to fp32 of partial sums."""
    return y.abs() * 2.0 ** -8 + x.shape[1] * 2.0 ** -24 * (x.abs() @ w.abs().t()) + 1e-30


# (rows, columns, K), edges of K and of strips among them (TILES below names tiles, and asserts that it runs them)
SHAPES = [
    (65, 16, 8), (97, 40, 72), (320, 768, 768), (129, 1000, 520), (257, 2048, 2056), (96, 6144, 768),
    (700, 1504, 1000), (193, 4100, 768), (320, 6144, 712),
    (1000, 3096, 2008), (1030, 6104, 264), (2100, 11264, 520),
    (2049, 2304, 768), (700, 6160, 776),
    (700, 17928, 1032),
]

# tile (rows, packed rows): (rows, packed rows, K) of products that run it, none of them whole tiles; K ends inside a step and with one
TILES = {
    (32, 32): [(97, 272, 136), (70, 272, 128)],
    (64, 64): [(193, 2320, 136), (97, 4112, 128)],
    (64, 128): [(130, 11280, 136), (450, 4112, 128), (450, 4112, 768)],
    (128, 128): [(321, 6160, 136), (193, 11280, 64), (321, 6160, 128)],
    (128, 192): [(700, 6160, 520), (1300, 3088, 768)],
    (256, 256): [(1025, 11280, 520), (700, 17936, 1032), (1025, 11280, 768)],
}


@pytest.mark.parametrize("tile,rows,packed,k", [(t, *s) for t, shapes in TILES.items() for s in shapes])
def test_every_tile_gives_the_same_bits(cuda, tile, rows, packed, k):
    """The sums do not depend on the tile: all epilogues, stored 16 bytes a lane and less, against the same rows in calls of 32 to 96 that run
    small tiles, and the plain product against 64 bits."""
    from ohara_amd import ops
    from ohara_amd._lib import check, lib

    of = lib().ohara_gemm_tile_of
    assert of(rows, packed, k) == 1000 * tile[0] + tile[1]
    step = 32 if tile == (64, 64) else 96
    assert tile == (32, 32) or of(step, packed, k) != 1000 * tile[0] + tile[1]
    g = torch.Generator(device=cuda).manual_seed(rows + packed + k)
    x = (torch.randn(rows, k, generator=g, device=cuda) * 3).to(BF)
    w = (torch.randn(packed, k, generator=g, device=cuda) * 0.3).to(BF)
    spans = [slice(r, min(r + step, rows)) for r in range(0, rows, step)]
    for n in (packed, packed - 8, packed - 5):
        wp, res = ops.pack_linear(w[:n].contiguous()), torch.randn(rows, n, generator=g, device=cuda).to(BF)
        got, summed = ops.gemm(x, wp), ops.gemm(x, wp, residual=res)
        assert torch.equal(got, torch.cat([ops.gemm(x[s], wp) for s in spans]))
        assert torch.equal(summed, torch.cat([ops.gemm(x[s], wp, residual=res[s]) for s in spans]))
        if n == packed - 5:
            want = x.double() @ w[:n].double().t()
            assert ((got.double() - want).abs() <= _bound(x.double(), w[:n].double(), want)).all()
        wide = torch.full((rows, n + 4), 7.0, dtype=BF, device=cuda)
        assert torch.equal(ops.gemm(x, wp, out=wide[:, :n]), got) and (wide[:, n:] == 7.0).all()
    for f in (packed // 2, packed // 2 - 3):
        gates = ops.pack_gate_up(w[:f].contiguous(), w[f:2 * f].contiguous())
        got = ops.gemm(x, gates)
        assert torch.equal(got, torch.cat([ops.gemm(x[s], gates) for s in spans]))
        wide = torch.full((rows, f + 4), 7.0, dtype=BF, device=cuda)
        assert torch.equal(ops.gemm(x, gates, out=wide[:, :f]), got) and (wide[:, f:] == 7.0).all()
    # rotary: heads of 16, an odd number of query heads; positions in a row, and given row by row
    H, D, T = packed // 16 - 2, 16, rows + 8
    ang = torch.rand(T, D // 2, generator=g, device=cuda) * 6.28
    cos, sin = ang.cos().to(BF), ang.sin().to(BF)
    wq = ops.pack_qkv(w[:H * D], w[H * D:H * D + D], w[H * D + D:])
    keys, values = (torch.full((4, T, 1, D), 9.0, dtype=BF, device=cuda) for _ in range(2))
    q = ops.qkv_rope_append(x, wq, None, 1e-5, H, 1, D, cos, sin, 3, keys[:1], values[:1], seq_len=rows)
    assert (keys[0, 3:3 + rows] != 9.0).any(-1).all() and (keys[0, :3] == 9.0).all() and (keys[0, 3 + rows:] == 9.0).all()
    by_row = torch.empty_like(q)

    def row_by_row(s, row):  # (always in tiles, also up to 64 rows)
        n = s.stop - s.start
        at = torch.cat([torch.arange(3 + s.start, 3 + s.stop), torch.full((n,), row)]).to(cuda, torch.int32)
        check(lib().ohara_qkv_rope_append_rows_bf16(x[s].data_ptr(), k, wq.data.data_ptr(), k, n, H, 1, D, cos.data_ptr(), sin.data_ptr(),
                                                    at.data_ptr(), by_row[s].data_ptr(), keys.data_ptr(), values.data_ptr(), T,
                                                    torch.cuda.current_stream().cuda_stream), "rows")

    for row, parts in ((1, [slice(0, rows)]), (3, spans)):
        by_row.zero_()
        for s in parts:
            row_by_row(s, row)
        assert torch.equal(by_row, q) and torch.equal(keys[row], keys[0]) and torch.equal(values[row], values[0])
    assert (keys[2] == 9.0).all() and (values[2] == 9.0).all()


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


# 32 x 32 tiles, 64 x 64, then 128 x 128 (K is short)
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


# width, depth, rows; the parts of the residual's product and of the one with two addends, and their tiles (1000 rows + columns)
PARTS = [
    (768, 3072, 65, (4, 32032), (4, 32032)), (768, 3072, 129, (4, 32032), (4, 32032)), (768, 3072, 400, (4, 64064), None),
    (768, 3072, 673, (2, 64064), None), (768, 3072, 1281, (2, 64128), None), (2048, 2048, 300, None, None), (2048, 2048, 410, (2, 64064), None),
    (2048, 5632, 33, (4, 32032), (4, 32032)), (2048, 5632, 192, (4, 64064), (4, 64064)), (2048, 5632, 401, (4, 128128), (4, 128128)),
    (2048, 5632, 1408, (2, 128192), (2, 128192)), (2048, 5632, 1500, (4, 256256), None), (2048, 5632, 3000, (2, 256256), None),
    (2560, 10240, 33, (8, 64064), (8, 64064)), (2560, 10240, 65, (8, 64128), (8, 64128)), (2560, 10240, 301, (8, 128128), (8, 128128)),
    (2560, 10240, 513, (8, 256256), (8, 256256)), (2560, 10240, 1000, (4, 128192), (4, 128192)), (2560, 10240, 2400, (2, 256256), (2, 256256)),
    (16, 4096, 97, (8, 32032), (8, 32032)), (4096, 4096, 70, (4, 64128), (4, 64128)), (4096, 4096, 228, (2, 64128), (2, 64128)),
    (4096, 14336, 986, (2, 128128), (2, 128128)),
]


@pytest.mark.parametrize("n,k,rows,residual,add2s", PARTS)
def test_products_in_parts_of_the_depth(cuda, n, k, rows, residual, add2s):
    """The residual product with the norm behind it, and the one with a bias and two addends, in parts of the depth against 64 bits: an
    fp32 sum of k products in any order, rounded where the products over the whole depth are; without room those are taken."""
    from ohara_amd import ops
    from ohara_amd._lib import check, lib

    g = torch.Generator(device=cuda).manual_seed(n + k + rows)
    x, w = (torch.randn(r, k, generator=g, device=cuda).to(torch.bfloat16) for r in (rows, n))
    res, add2 = (torch.randn(rows, n, generator=g, device=cuda).to(torch.bfloat16) for _ in range(2))
    bias, norm = (torch.randn(n, generator=g, device=cuda).to(torch.bfloat16) for _ in range(2))
    y, mass = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    sum_err = mass * k * 2.0 ** -24
    packed, stream = ops.pack_linear(w), torch.cuda.current_stream().cuda_stream

    def half(v, e):  # a value known to e, rounded to bf16: its error
        return e + (v.abs() + e) * 2.0 ** -8

    y_err = half(y, sum_err)
    want, want_err = res.double() + y, half(res.double() + y, y_err)
    room = lib().ohara_gemm_residual_norm_bytes(rows, n, k)
    for size, parts in ((room, residual), (lib().ohara_linear_bias_add2_bytes(rows, n, k), add2s)):
        assert size == (4 * parts[0] * rows * n if parts else 0)
        assert not parts or lib().ohara_gemm_tile_of(rows, n * parts[0], k // parts[0]) == parts[1]
    for size in {room, 0}:
        ws = torch.full((size + 64,), 0xFF, dtype=torch.uint8, device=cuda)
        out, xn = res.clone(), torch.empty_like(res)
        check(lib().ohara_gemm_residual_norm_bf16(x.data_ptr(), k, packed.data.data_ptr(), n, k, rows, out.data_ptr(), norm.data_ptr(), 1e-5,
                                                  xn.data_ptr(), ws.data_ptr(), size, stream), "residual_norm")
        assert ((out.double() - want).abs() <= want_err).all()
        o = out.double()
        v = o / (o.square().mean(-1, keepdim=True) + 1e-5).sqrt()
        assert ((xn.double() - v * norm.double()).abs() <= (v * norm.double()).abs() * 2.0 ** -7 + 1e-6).all()  # rounded twice
        assert (ws[size:] == 0xFF).all()
        plain = res.clone()
        check(lib().ohara_gemm_residual_norm_bf16(x.data_ptr(), k, packed.data.data_ptr(), n, k, rows, plain.data_ptr(), None, 1e-5, None,
                                                  ws.data_ptr(), size, stream), "residual_norm")
        assert torch.equal(plain, out)
    with_bias = y + bias.double()
    b_err = half(with_bias, sum_err)
    first, first_err = with_bias + res.double(), half(with_bias + res.double(), b_err)
    total, total_err = first + add2.double(), half(first + add2.double(), first_err)
    got = ops.linear_bias(x, packed, bias, "add2", add1=res, add2=add2)
    assert ((got.double() - total).abs() <= total_err).all()
    odd = torch.empty(rows, n + 4, dtype=torch.bfloat16, device=cuda)[:, 4:]  # not on 16 bytes: over the whole depth
    ops.linear_bias(x, packed, bias, "add2", add1=res, add2=add2, out=odd)
    assert ((odd.double() - total).abs() <= total_err).all()


def test_rows_far_apart_are_multiplied_whole(cuda):
    """Rows whose distance the parts of the depth do not address (views into very wide buffers) take the product over the whole depth."""
    from ohara_amd import ops
    from ohara_amd._lib import check, lib

    ldx = 1 << 23  # 2^23 elements: a tile of 256 such rows is 4 GiB
    rows, far = 33, torch.empty(33 * ldx, dtype=torch.bfloat16, device=cuda)
    g = torch.Generator(device=cuda).manual_seed(1)
    for n, k in ((2560, 10240), (2048, 5632)):
        assert lib().ohara_linear_bias_add2_bytes(rows, n, k) > 0 and lib().ohara_gemm_residual_norm_bytes(rows, n, k) > 0
        x, w = (torch.randn(r, k, generator=g, device=cuda).to(torch.bfloat16) for r in (rows, n))
        a1, a2 = (torch.randn(rows, n, generator=g, device=cuda).to(torch.bfloat16) for _ in range(2))
        bias, norm = (torch.randn(n, generator=g, device=cuda).to(torch.bfloat16) for _ in range(2))
        wide = far.view(rows, ldx)[:, :k]
        wide.copy_(x)
        packed, stream = ops.pack_linear(w), torch.cuda.current_stream().cuda_stream
        whole = torch.empty(rows, n + 4, dtype=torch.bfloat16, device=cuda)[:, 4:]  # (not on 16 bytes: over the whole depth too)
        ops.linear_bias(x, packed, bias, "add2", add1=a1, add2=a2, out=whole)
        assert torch.equal(ops.linear_bias(wide, packed, bias, "add2", add1=a1, add2=a2), whole)
        out, xn = a1.clone(), torch.empty_like(a1)
        ws = torch.empty(lib().ohara_gemm_residual_norm_bytes(rows, n, k), dtype=torch.uint8, device=cuda)
        check(lib().ohara_gemm_residual_norm_bf16(wide.data_ptr(), ldx, packed.data.data_ptr(), n, k, rows, out.data_ptr(), norm.data_ptr(), 1e-5,
                                                  xn.data_ptr(), ws.data_ptr(), ws.numel(), stream), "residual_norm")
        want = ops.gemm_skinny(x, packed, residual=a1, out=a1.clone())
        assert torch.equal(out, want) and torch.equal(xn, ops.rmsnorm(want, norm))
