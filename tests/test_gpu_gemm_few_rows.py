"""The tiles of fewer than 1024 rows that carry an epilogue or a part of the depth: edges of rows, strips and K, against the same rows in calls of 32 that
run small tiles, bit for bit (the sums do not depend on the tile); parts against 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

# tile, rows, packed rows, K (a step and a piece, whole steps, an edge inside the last one)
CASES = [
    (48064, 35, 8208, 520), (48064, 97, 4112, 2056), (80064, 65, 8208, 776), (80064, 193, 4112, 1032), (96064, 65, 17936, 72), (96064, 400, 6160, 2056),
    (96096, 65, 17936, 520), (96096, 130, 11280, 1032), (128096, 97, 17936, 520), (128096, 193, 11280, 1032), (64064, 300, 3088, 1032),
    (128128, 161, 17936, 72), (128128, 600, 11280, 520), (128128, 193, 17936, 520), (128192, 700, 11280, 520), (192128, 900, 6160, 520), (192128, 900, 6160, 1032),
    # in halves
    (128193, 193, 17936, 776), (128193, 450, 11280, 1032), (128257, 300, 17936, 1032), (128257, 513, 11280, 2056), (256257, 700, 17936, 1032), (256257, 1000, 11280, 2056), (128193, 700, 11280, 2560),
]


@pytest.mark.parametrize("tile,rows,packed,k", CASES)
def test_residual_and_gated(cuda, tile, rows, packed, k):
    from ohara_amd import ops
    from ohara_amd._lib import lib

    with_ = lib().ohara_gemm_tile_with
    assert with_(rows, packed, k, 1, 1) == with_(rows, packed, k, 2, 1) == tile and with_(32, packed, k, 1, 1) != tile
    g = torch.Generator(device=cuda).manual_seed(rows + packed + k)
    x = (torch.randn(rows, k, generator=g, device=cuda) * 3).to(BF)
    w = (torch.randn(packed, k, generator=g, device=cuda) * 0.3).to(BF)
    w[5, k - 1] = float("inf")  # (past K the walk stands in other values: none of them may be multiplied, not even by zero)
    x[:, k - 1] = x[:, k - 1].abs() + 1
    spans = [slice(r, min(r + 32, rows)) for r in range(0, rows, 32)]
    for n in (packed, packed - 5):
        wp, res = ops.pack_linear(w[:n].contiguous()), torch.randn(rows, n, generator=g, device=cuda).to(BF)
        assert torch.equal(ops.gemm(x, wp, residual=res), torch.cat([ops.gemm(x[s], wp, residual=res[s]) for s in spans]))
    for f in (packed // 2, packed // 2 - 3):
        gates = ops.pack_gate_up(w[:f].contiguous(), w[f:2 * f].contiguous())
        assert torch.equal(ops.gemm(x, gates), torch.cat([ops.gemm(x[s], gates) for s in spans]))


# ... of a vocabulary's plain store, whose other products run the tile of ohara_gemm_tile_of
@pytest.mark.parametrize("tile,rows,packed,k", [(96064, 66, 32016, 2056), (96096, 66, 20016, 776), (128096, 97, 20016, 776), (192128, 192, 32016, 1032), (128193, 193, 20016, 776),
                                                (128257, 193, 32016, 1032), (128192, 300, 32016, 1032), (256257, 385, 32016, 1032), (256257, 700, 20016, 768)])
def test_vocabulary(cuda, tile, rows, packed, k):
    from ohara_amd import ops
    from ohara_amd._lib import lib

    assert lib().ohara_gemm_tile_with(rows, packed, k, 0, 1) == tile
    assert lib().ohara_gemm_tile_with(rows, 17936, k, 0, 1) == lib().ohara_gemm_tile_of(rows, 17936, k) + (lib().ohara_gemm_tile_of(rows, 17936, k) == 256256)
    g = torch.Generator(device=cuda).manual_seed(rows + packed + k)
    x = (torch.randn(rows, k, generator=g, device=cuda) * 3).to(BF)
    w = (torch.randn(packed, k, generator=g, device=cuda) * 0.3).to(BF)
    for n in (packed, packed - 5):
        wp = ops.pack_linear(w[:n].contiguous())
        assert torch.equal(ops.gemm(x, wp), torch.cat([ops.gemm(x[r:r + 32], wp) for r in range(0, rows, 32)]))


# tile, head width, query heads, key heads, sequences, positions of each, K
ROTARY = [
    (48064, 48, 10, 2, 3, 267, 1032), (80064, 128, 16, 4, 1, 341, 1032), (96064, 128, 16, 4, 2, 228, 2056), (96096, 80, 32, 32, 2, 136, 2056),
    (96096, 128, 16, 4, 13, 51, 520), (128096, 64, 16, 16, 1, 962, 1032), (128192, 128, 32, 8, 3, 221, 520), (128128, 128, 32, 8, 5, 197, 136),
    (128193, 128, 32, 8, 3, 221, 2056), (128257, 48, 64, 64, 2, 350, 1032), (256257, 128, 32, 32, 2, 450, 1032),
]


@pytest.mark.parametrize("tile,D,H,Hkv,B,S,k", ROTARY)
def test_rotary(cuda, tile, D, H, Hkv, B, S, k):
    from ohara_amd import ops
    from ohara_amd._lib import lib

    assert lib().ohara_gemm_tile_with(B * S, (H + 2 * Hkv) * D, k, 3, 1) == tile
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


@pytest.mark.parametrize("d,ff,B,S,tile", [(2560, 10240, 1, 97, 128096), (1280, 5120, 2, 300, 128192), (1024, 4096, 1, 257, 96096), (768, 3072, 3, 200, 128128),
                                           (2560, 10240, 1, 65, 96096), (1280, 5120, 1, 130, 64064), (2560, 10240, 1, 200, 128193),
                                           (2560, 10240, 2, 150, 128257), (2048, 8192, 2, 400, 256257)])
def test_phi_input(cuda, d, ff, B, S, tile):
    from ohara_amd import ops
    from ohara_amd._lib import lib

    assert lib().ohara_gemm_tile_with(B * S, 3 * d + ff, d, 7, 1) == tile
    pos, g = 3, torch.Generator(device=cuda).manual_seed(7)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda).to(BF)  # noqa: E731
    x, bias, w = r(B * S, d), r(3 * d + ff), ops.pack_linear((r(3 * d + ff, d).float() * 0.1).to(BF))

    def run(step):
        kc, vc = (torch.full((B, S + 5, 8, d // 8), 9.0, dtype=BF, device=cuda) for _ in range(2))
        q, act = torch.empty(B * S, d, dtype=BF, device=cuda), torch.empty(B * S, ff, dtype=BF, device=cuda)
        for b in range(B) if step < S else [0]:
            for a in range(0, max(S - step, 0) + 1, step):
                n = step if a + 2 * step <= S else S - a  # (64 rows and fewer may be summed by waves)
                at = slice(b * S + a, b * S + a + n) if step < S else slice(0, B * S)
                seqs = slice(b, b + 1) if step < S else slice(0, B)
                ops.phi_block_in(x[at], None, None, 1e-5, w, bias, d, ff, 1 if step < S else B, n, pos + a, kc[seqs], vc[seqs], q[at], act[at])
        return q, act, kc, vc

    assert all(torch.equal(a, b) for a, b in zip(run(S), run(65)))


# tile, columns, depth, rows, parts
@pytest.mark.parametrize("tile,n,k,rows,parts", [
    (48064, 2048, 5632, 82, 4), (80064, 2048, 5632, 131, 4), (80064, 768, 3072, 719, 2), (96064, 2048, 5632, 257, 4), (96096, 2560, 10240, 68, 8), (96096, 1536, 4096, 341, 4),
    (128096, 2560, 10240, 103, 8), (128193, 2048, 5632, 516, 4), (128257, 2560, 10240, 700, 4), (256257, 2560, 10240, 1000, 4), (192128, 2048, 5632, 642, 4), (64064, 2048, 5632, 103, 4), (128128, 2048, 5632, 390, 4),
])
def test_parts_of_the_depth(cuda, tile, n, k, rows, parts):
    from ohara_amd._lib import check, lib
    from ohara_amd import ops

    room = lib().ohara_gemm_residual_norm_bytes(rows, n, k)
    assert room == 4 * parts * rows * n and lib().ohara_gemm_tile_with(rows, n, k, 1, parts) == tile
    g = torch.Generator(device=cuda).manual_seed(n + k + rows)
    x, w, res = (torch.randn(*s, generator=g, device=cuda).to(BF) for s in ((rows, k), (n, k), (rows, n)))
    xd, wd = x.double(), w.double()
    y = xd @ wd.t()
    # k roundings to fp32 of partial sums, one of the product to bf16 and one of the sum with the residual
    bound = (xd.abs() @ wd.abs().t()) * k * 2.0 ** -24 + y.abs() * 2.0 ** -8
    bound = bound * 1.01 + (y + res.double()).abs() * 2.0 ** -8 + bound * 2.0 ** -8
    ws, out = torch.full((room + 64,), 0xFF, dtype=torch.uint8, device=cuda), res.clone()
    check(lib().ohara_gemm_residual_norm_bf16(x.data_ptr(), k, ops.pack_linear(w).data.data_ptr(), n, k, rows, out.data_ptr(), None, 1e-5, None,
                                              ws.data_ptr(), room, torch.cuda.current_stream().cuda_stream), "residual_norm")
    assert ((out.double() - (y + res.double())).abs() <= bound).all()
    assert (ws[room:] == 0xFF).all()


# rows, columns, depth, parts, a tile that would make a round of workgroups if it reached from one part into the next
@pytest.mark.parametrize("rows,n,k,parts,across", [(375, 2640, 11264, 8, 128256), (618, 3200, 9216, 4, 128256), (213, 672, 9216, 8, 80064), (375, 784, 4096, 4, 80064),
                                                   (364, 1984, 6144, 8, 128192), (412, 656, 4096, 4, 80064)])
def test_parts_are_counted_by_themselves(cuda, rows, n, k, parts, across):
    from ohara_amd._lib import lib

    strips, height, width = n // 16, across // 1000, across % 1000 // 16
    down = -(-rows // height)
    assert down * -(-strips * parts // width) <= 256 < down * -(-strips // width) * parts
    assert lib().ohara_gemm_tile_with(rows, n, k, 1, parts) // 2 * 2 != across


# rows, packed rows, depth, epilogue, parts, the tile: a round of 64 x 48, and 260, 264 and 268 of 64 x 128
@pytest.mark.parametrize("rows,packed,k,epilogue,parts,tile", [(45, 10272, 1920, 2, 1, 64048), (136, 3872, 1600, 1, 1, 64048), (47, 9216, 1536, 3, 1, 64048), (44, 1408, 5120, 1, 8, 64048),
                                                               (217, 8272, 2528, 7, 1, 128096), (217, 8384, 1280, 2, 1, 128096), (206, 8528, 816, 7, 1, 96064)])
def test_tiles_that_stay(cuda, rows, packed, k, epilogue, parts, tile):
    from ohara_amd._lib import lib

    assert lib().ohara_gemm_tile_with(rows, packed, k, epilogue, parts) == tile
