"""The tiles whose waves work in two halves, those that fill the chip once with few rows, the rotary epilogue by whole rows of the tables,
and rows in two launches:
depths that end inside a step, with one and before the ring is full, against the same rows in calls of 32 that run small tiles, bit for bit, and against 64 bits; rotated rows
against the plain product's, rotated here."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

# tile, rows, packed rows, K: one step, a step and a piece, less than the ring, every remainder of 64 that counts (8, 32, 40, 0)
CASES = [
    (128192, 1025, 4512, 64), (128192, 1025, 4512, 72), (128192, 1025, 4512, 128), (128192, 1025, 4400, 168), (128192, 1100, 4400, 264),
    (128192, 1024, 6144, 776), (128256, 1025, 6944, 136), (128256, 3000, 2320, 328), (128256, 2049, 3088, 520), (128256, 1537, 4112, 544),
    (128256, 2049, 3088, 768), (256256, 1025, 12720, 72), (256256, 1025, 11760, 168), (256256, 1100, 11280, 192), (256256, 1025, 11280, 200),
    (256256, 2049, 6160, 296), (256256, 2049, 6160, 320), (256256, 1537, 8208, 360),
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


def _parts(rows, step=96):
    """Calls of few rows (more than 64: in tiles too), the last one with what is left as well."""
    at = list(range(0, rows - 2 * step, step))
    return [slice(a, a + step) for a in at] + [slice((at[-1] if at else -step) + step, rows)]


EPILOGUES = {"plain": 0, "residual": 1, "swiglu": 2, "bias": 4, "gelu": 5, "add2": 6, "softcap": 8, "lookup": 9, "xielu": 11}


@pytest.mark.parametrize("rows,n,k,two", [(4500, 4048, 832, True), (1300, 11936, 1032, True), (4500, 4112, 200, False), (3000, 6160, 200, False), (4500, 11280, 136, False)])
def test_rows_in_two_launches(cuda, rows, n, k, two):
    """Whole rounds of large tiles and the rest by itself (short depths: all in one): every epilogue finds the rest's rows."""
    from ohara_amd import ops
    from ohara_amd._lib import lib

    for name, epilogue in EPILOGUES.items():
        first = lib().ohara_gemm_first_rows(rows, n, k, epilogue, 0)
        assert 0 < first < rows and first % 256 == 0 if two else first == 0, name

    g = torch.Generator(device=cuda).manual_seed(rows + n)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda).to(BF)  # noqa: E731
    x, w, bias, res, add2, table = r(rows, k), r(n, k), r(n), r(rows, n), r(rows, n), r(50, n + 8)
    ids = torch.randint(0, 50, (rows,), generator=g, device=cuda)
    wp, gates = ops.pack_linear(w), ops.pack_gate_up(w[:n // 2].contiguous(), w[n // 2:].contiguous())
    calls = {
        "plain": lambda s: ops.gemm(x[s], wp), "residual": lambda s: ops.gemm(x[s], wp, residual=res[s]), "swiglu": lambda s: ops.gemm(x[s], gates),
        "bias": lambda s: ops.linear_bias(x[s], wp, bias), "gelu": lambda s: ops.linear_bias(x[s], wp, bias, "gelu"),
        "add2": lambda s: ops.linear_bias(x[s], wp, bias, "add2", add1=res[s], add2=add2[s]), "softcap": lambda s: ops.gemm_softcap(x[s], wp, 20.0),
        "lookup": lambda s: ops.gemm_gelu_lookup(x[s], wp, table, 8, ids[s]), "xielu": lambda s: ops.gemm_xielu(x[s], wp, bias, 0.3, 0.2),
    }
    for name, call in calls.items():
        assert torch.equal(call(slice(0, rows)), torch.cat([call(s) for s in _parts(rows)])), name


@pytest.mark.parametrize("B,S,H,Hkv,D,k,two", [(2, 1050, 58, 2, 128, 768, True), (2, 1050, 118, 2, 64, 768, True), (2, 1050, 162, 2, 48, 768, True),
                                               (2, 2250, 240, 8, 16, 136, False), (3, 1500, 48, 8, 64, 136, False), (3, 1000, 32, 8, 64, 520, False)])
def test_rotary_rows_in_two_launches(cuda, B, S, H, Hkv, D, k, two):
    from ohara_amd import ops
    from ohara_amd._lib import check, lib

    assert (0 < lib().ohara_gemm_first_rows(B * S, (H + 2 * Hkv) * D, k, 3, D) < B * S) == two

    g = torch.Generator(device=cuda).manual_seed(S + D)
    rows, pos, T = B * S, 3, S + 5
    x = torch.randn(rows, k, generator=g, device=cuda).to(BF)
    w = (torch.randn((H + 2 * Hkv) * D, k, generator=g, device=cuda) * 0.1).to(BF)
    ang = torch.rand(T, D // 2, generator=g, device=cuda) * 6.28
    cos, sin = ang.cos().to(BF), ang.sin().to(BF)
    wq = ops.pack_qkv(w[:H * D], w[H * D:(H + Hkv) * D], w[(H + Hkv) * D:])
    y = ops.gemm(x, ops.pack_linear(w)).view(B, S, H + 2 * Hkv, D)
    e, o = y[..., 0::2].float(), y[..., 1::2].float()
    c, n = (t[pos:pos + S].float().view(1, S, 1, D // 2) for t in (cos, sin))
    turned = torch.stack([e * c - o * n, e * n + o * c], -1).flatten(-2).to(BF)
    keys, values = (torch.full((B + 1, T, Hkv, D), 9.0, dtype=BF, device=cuda) for _ in range(2))
    q = ops.qkv_rope_append(x, wq, None, 1e-5, H, Hkv, D, cos, sin, pos, keys[:B], values[:B], seq_len=S)
    assert torch.equal(q.view(B, S, H, D), turned[:, :, :H]) and torch.equal(keys[:B, pos:pos + S], turned[:, :, H:H + Hkv])
    assert torch.equal(values[:B, pos:pos + S], y[:, :, H + Hkv:])
    q2, k2, v2 = ops.qkv_rope(x, wq, None, 1e-5, H, Hkv, D, cos, sin, pos, T, seq_len=S)
    assert torch.equal(q2, q) and torch.equal(k2.view(B, S, Hkv, D), turned[:, :, H:H + Hkv]) and torch.equal(v2.view(B, S, Hkv, D), y[:, :, H + Hkv:])
    # positions given row by row, the sequences' rows of the cache in another order
    at = torch.cat([torch.arange(pos, pos + S).repeat(B), torch.arange(B, 0, -1).repeat_interleave(S)]).to(cuda, torch.int32)
    keys2, values2, q3 = torch.full_like(keys, 9.0), torch.full_like(values, 9.0), torch.empty_like(q)
    check(lib().ohara_qkv_rope_append_rows_bf16(x.data_ptr(), k, wq.data.data_ptr(), k, rows, H, Hkv, D, cos.data_ptr(), sin.data_ptr(), at.data_ptr(),
                                                q3.data_ptr(), keys2.data_ptr(), values2.data_ptr(), T, torch.cuda.current_stream().cuda_stream), "rows")
    assert torch.equal(q3, q) and (keys2[0] == 9.0).all()
    assert all(torch.equal(keys2[B - b], keys[b]) and torch.equal(values2[B - b], values[b]) for b in range(B))


@pytest.mark.parametrize("d,ff,two", [(768, 1792, True), (512, 2576, False)])
def test_phi_rows_in_two_launches(cuda, d, ff, two):
    from ohara_amd import ops
    from ohara_amd._lib import lib

    B, S, pos = 2, 2250, 3
    assert (0 < lib().ohara_gemm_first_rows(B * S, 3 * d + ff, d, 7, 0) < B * S) == two
    g = torch.Generator(device=cuda).manual_seed(7)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda).to(BF)  # noqa: E731
    x, bias, w = r(B * S, d), r(3 * d + ff), ops.pack_linear((r(3 * d + ff, d).float() * 0.1).to(BF))

    def run(step):
        kc, vc = (torch.full((B, S + 5, 8, d // 8), 9.0, dtype=BF, device=cuda) for _ in range(2))
        q, act = torch.empty(B * S, d, dtype=BF, device=cuda), torch.empty(B * S, ff, dtype=BF, device=cuda)
        if step == S:
            ops.phi_block_in(x, None, None, 1e-5, w, bias, d, ff, B, S, pos, kc, vc, q, act)
        else:
            for b in range(B):
                for s in _parts(S, step):
                    at = slice(b * S + s.start, b * S + s.stop)
                    ops.phi_block_in(x[at], None, None, 1e-5, w, bias, d, ff, 1, s.stop - s.start, pos + s.start, kc[b:b + 1], vc[b:b + 1], q[at], act[at])
        return q, act, kc, vc

    assert all(torch.equal(a, b) for a, b in zip(run(S), run(96)))
