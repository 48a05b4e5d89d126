"""More large tiles than CUs at depths of whole steps, where a workgroup goes from tile to tile with its loads ahead of it: every tile in halves, depths of
three steps and more, last tiles that are not whole, CUs with a tile less than others, against the same rows in calls of few that run small
tiles, bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

# tile, rows, packed rows, K
CASES = [(256256, 4763, 6160, 192), (256256, 5762, 5136, 192), (256256, 6761, 6160, 256), (256256, 4096, 6144, 768), (128256, 6428, 2320, 256), (128256, 6428, 2320, 320),
         (128256, 3764, 6160, 256), (128192, 5096, 2064, 192), (128192, 2099, 5136, 192), (128192, 5429, 1552, 512)]


def _parts(rows, step=96):
    """Calls of few rows (more than 64: in tiles too), the last one with what is left as well."""
    at = list(range(0, rows - 2 * step, step))
    return [slice(a, a + step) for a in at] + [slice(at[-1] + step, rows)]


@pytest.mark.parametrize("tile,rows,packed,k", CASES)
def test_rounds(cuda, tile, rows, packed, k):
    from ohara_amd import ops
    from ohara_amd._lib import lib

    tm, tn = tile // 1000, tile % 1000
    assert -(-rows // tm) * -(-packed // tn) > 256 and (lib().ohara_gemm_tile_of(rows, packed, k) == tile or (rows, packed, k) == (4096, 6144, 768))
    g = torch.Generator(device=cuda).manual_seed(rows + packed + k)
    x = (torch.randn(rows, k, generator=g, device=cuda) * 3).to(BF)
    w = (torch.randn(packed, k, generator=g, device=cuda) * 0.3).to(BF)
    for n in (packed, packed - 5):
        wp, res = ops.pack_linear(w[:n].contiguous()), torch.randn(rows, n, generator=g, device=cuda).to(BF)
        small, summed = ([ops.gemm(x[s], wp, residual=r) for s, r in ((s, res[s] if with_ else None) for s in _parts(rows))] for with_ in (False, True))
        for _ in range(2):
            assert torch.equal(ops.gemm(x, wp), torch.cat(small))
            assert torch.equal(ops.gemm(x, wp, residual=res), torch.cat(summed))
    f = packed // 2
    gates = ops.pack_gate_up(w[:f].contiguous(), w[f:2 * f].contiguous())
    assert torch.equal(ops.gemm(x, gates), torch.cat([ops.gemm(x[s], gates) for s in _parts(rows)]))


@pytest.mark.parametrize("rows,n,k", [(4763, 6160, 320), (4763, 6160, 1536)])
def test_every_epilogue(cuda, rows, n, k):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(rows + n)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda).to(BF)  # noqa: E731
    x, w, bias, res, add2, table = r(rows, k), r(n, k), r(n), r(rows, n), r(rows, n), r(50, n + 8)
    ids = torch.randint(0, 50, (rows,), generator=g, device=cuda)
    wp = ops.pack_linear(w)
    for call in (
        lambda s: ops.linear_bias(x[s], wp, bias), lambda s: ops.linear_bias(x[s], wp, bias, "gelu"),
        lambda s: ops.linear_bias(x[s], wp, bias, "add2", add1=res[s], add2=add2[s]), lambda s: ops.gemm_softcap(x[s], wp, 20.0),
        lambda s: ops.gemm_gelu_lookup(x[s], wp, table, 8, ids[s]), lambda s: ops.gemm_xielu(x[s], wp, bias, 0.3, 0.2),
    ):
        assert torch.equal(call(slice(0, rows)), torch.cat([call(s) for s in _parts(rows)]))


@pytest.mark.parametrize("B,S,H,Hkv,D,k", [(2, 2548, 40, 4, 128, 192), (5, 1240, 80, 8, 64, 320), (1, 5096, 44, 2, 128, 768)])
def test_rotary(cuda, B, S, H, Hkv, D, k):
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
    assert (keys[:, :pos] == 9.0).all() and (keys[:, pos + S:] == 9.0).all()
