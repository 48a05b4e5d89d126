"""Projections of up to 64 normed rows where several strips share a workgroup, and where eight waves share a strip: edges of K, of rows
and of strips, against the norm and the projection as two calls."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _check(got, x, w, nw, eps, plain):
    """`plain`: the projection of rows normed before.  Only the two fp32 sums (of the squares, over K) are in another order: a normed value
    may round to its neighbour (2^-8 of it at most), a result likewise."""
    from ohara_amd import ops

    xn = ops.rmsnorm(x, nw, eps).double()
    mass = xn.abs() @ w.double().abs().t()
    assert ((got.double() - xn @ w.double().t()).abs() <= (xn @ w.double().t()).abs() * 2.0 ** -8 + mass * (2.0 ** -8 + x.shape[1] * 2.0 ** -24)).all()
    assert (got != plain).float().mean() <= 0.05


# (columns, K): two, three and four strips a workgroup with eight waves (K up to 1024) and with sixteen, the last group not full; then one strip
# with eight waves; then more strips than groups take, where rows that wide_kernel cannot hold have a strip and four waves
SHAPES = [(4112, 8), (8200, 1000), (12304, 1024), (4128, 1032), (11264, 2048), (12000, 1544), (16368, 2040), (3072, 2048), (40, 1032),
          (16400, 1032), (16416, 2048)]


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 64])
def test_store_and_gates(cuda, rows, n, k):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(rows + n + k)
    x = (torch.randn(rows, k, generator=g, device=cuda) * torch.logspace(-2, 2, rows, device=cuda)[:, None]).to(BF)
    nw = (1 + 0.3 * torch.randn(k, generator=g, device=cuda)).to(BF)
    w = (torch.randn(n, k, generator=g, device=cuda) * 0.05).to(BF)
    packed, xn = ops.pack_linear(w), ops.rmsnorm(x, nw, 1e-5)
    _check(ops.gemm_skinny(x, packed, nw, 1e-5), x, w, nw, 1e-5, ops.gemm_skinny(xn, packed))
    f = n // 2
    gates = ops.pack_gate_up(w[:f], w[f:2 * f])
    got, plain = ops.gemm_skinny(x, gates, nw, 1e-5), ops.gemm_skinny(xn, gates)
    assert (got != plain).float().mean() <= 0.05
    gate, up = (xn.double() @ t.double().t() for t in (w[:f], w[f:2 * f]))
    mass_g, mass_u = (xn.double().abs() @ t.double().abs().t() for t in (w[:f], w[f:2 * f]))
    silu = gate * torch.sigmoid(gate)
    rel = 2.0 ** -8 + k * 2.0 ** -24
    # three roundings of the product's factors and itself, the gate's through a slope of at most 1.1, and neighbours in the normed rows
    bound = 1.02 * (silu.abs() * (up.abs() * 3 * 2.0 ** -8 + mass_u * rel) + 1.1 * (gate.abs() * 2.0 ** -8 + mass_g * rel) * (up.abs() + mass_u * rel))
    assert ((got.double() - silu * up).abs() <= bound + 1e-30).all()


@pytest.mark.parametrize("B,H,Hkv,D,K", [(1, 40, 8, 128, 1024), (17, 33, 33, 64, 776), (40, 48, 8, 64, 2048), (64, 16, 4, 128, 2048), (16, 16, 4, 128, 1288)])
def test_rotary(cuda, B, H, Hkv, D, K):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(B + K)
    x = torch.randn(B, K, generator=g, device=cuda).to(BF)
    nw = (1 + 0.3 * torch.randn(K, generator=g, device=cuda)).to(BF)
    ws = [(torch.randn(n * D, K, generator=g, device=cuda) * 0.05).to(BF) for n in (H, Hkv, Hkv)]
    ang = torch.rand(16, D // 2, generator=g, device=cuda) * 6.28
    cos, sin = ang.cos().to(BF), ang.sin().to(BF)
    wp, out = ops.pack_qkv(*ws), []
    for rows, norm in ((x, nw), (ops.rmsnorm(x, nw, 1e-5), None)):
        kc, vc = (torch.full((B, 16, Hkv, D), 9.0, dtype=BF, device=cuda) for _ in range(2))
        q = ops.qkv_rope_append(rows, wp, norm, 1e-5, H, Hkv, D, cos, sin, 5, kc, vc)
        assert (kc[:, :5] == 9.0).all() and (kc[:, 6:] == 9.0).all() and (vc[:, 6:] == 9.0).all()
        out.append((q, kc[:, 5].reshape(B, -1), vc[:, 5].reshape(B, -1)))
    _check(out[0][2], x, ws[2], nw, 1e-5, out[1][2])
    for got, plain in zip(*out):  # the rotation adds two values that may each be a neighbour
        assert (got != plain).float().mean() <= 0.05
        assert (got.float() - plain.float()).abs().max() <= 2.0 ** -6 * plain.float().abs().max()


@pytest.mark.parametrize("n,k", [(40, 760), (2304, 768), (2304, 776), (40, 1528), (2312, 1536), (2304, 1544), (4112, 768), (4112, 776), (8200, 1536), (8200, 1544)])
@pytest.mark.parametrize("rows", [1, 17, 40])
def test_shares_of_three_and_six_steps(cuda, rows, n, k):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(rows + n + k)
    x = torch.randn(rows, k, generator=g, device=cuda).to(BF)
    nw = (1 + 0.3 * torch.randn(k, generator=g, device=cuda)).to(BF)
    w = (torch.randn(n, k, generator=g, device=cuda) * 0.05).to(BF)
    packed = ops.pack_linear(w)
    _check(ops.gemm_skinny(x, packed, nw, 1e-5), x, w, nw, 1e-5, ops.gemm_skinny(ops.rmsnorm(x, nw, 1e-5), packed))


@pytest.mark.parametrize("n,k", SHAPES + [(4112, 576), (8200, 1352), (2304, 520)])
@pytest.mark.parametrize("rows", [1, 17, 40])
def test_infinite_weights_of_the_last_columns(cuda, rows, n, k):
    """Waves whose share of K ends early, or that have none: an infinite weight makes its own column infinite and no NaN."""
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(8)
    x = torch.rand(rows, k, generator=g, device=cuda).add_(0.5).to(BF)
    nw = torch.ones(k, device=cuda, dtype=BF)
    w = torch.randn(n, k, generator=g, device=cuda).to(BF)
    w[3, k - 1], w[n - 2, k - 8] = float("inf"), -float("inf")
    got = ops.gemm_skinny(x, ops.pack_linear(w), nw, 1e-5)
    assert (got[:, 3] == float("inf")).all() and (got[:, n - 2] == -float("inf")).all()
    rest = [c for c in range(n) if c not in (3, n - 2)]
    assert got[:, rest].isfinite().all()


@pytest.mark.parametrize("n,k", [(11264, 2048), (3072, 2048), (16416, 1032), (7680, 2560), (512, 2056)])
@pytest.mark.parametrize("rows", [17, 33, 64])
def test_norm_inside_the_projection_at_wide_models(cuda, rows, n, k):
    """Python norms these rows ahead of the product where the rule says so (from 33 rows here, from 17 past 2048 columns); a caller without
    room for normed rows (the last rows' logits of a batch) gets the kernels that norm them themselves."""
    from ohara_amd import _lib, ops

    assert _lib.lib().ohara_projection_norm_ahead(rows, k, n) == (rows > (16 if k > 2048 else 32))

    g = torch.Generator(device=cuda).manual_seed(rows + n)
    x, nw = torch.randn(rows, k, generator=g, device=cuda).to(BF), (1 + 0.3 * torch.randn(k, generator=g, device=cuda)).to(BF)
    w = (torch.randn(n, k, generator=g, device=cuda) * 0.05).to(BF)
    packed, out = ops.pack_linear(w), torch.empty(rows, n, dtype=BF, device=cuda)
    _lib.check(_lib.lib().ohara_gemm_skinny_bf16(x.data_ptr(), k, packed.data.data_ptr(), n, k, nw.data_ptr(), 1e-5, rows, _lib.EPI_STORE, None, 0,
                                                 out.data_ptr(), n, torch.cuda.current_stream().cuda_stream), "gemm_skinny")
    _check(out, x, w, nw, 1e-5, ops.gemm_skinny(x, packed, nw, 1e-5))


@pytest.mark.parametrize("H,G,K", [(4, 2, 1032), (24, 12, 2056)])
@pytest.mark.parametrize("batch,seq", [(17, 1), (64, 1), (3, 11), (1, 16), (1, 17)])
def test_rotary_rows_around_the_change_of_kernel(cuda, batch, seq, H, G, K):
    """Rows 16 | 17 at wide models: the same rows one sequence at a time (strips) and together, in tiles from 17 on where the projection is
    wide too, in strips where it is narrow."""
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(batch + seq)
    D, T, pos = 64, 40, 5
    x, nw = torch.randn(batch * seq, K, generator=g, device=cuda).to(BF), (1 + 0.3 * torch.randn(K, generator=g, device=cuda)).to(BF)
    wqkv = ops.pack_qkv(*((torch.randn(h * D, K, generator=g, device=cuda) * 0.05).to(BF) for h in (H, G, G)))
    angle = torch.rand(2 * T, D // 2, generator=g, device=cuda)
    cos, sin = angle.cos().to(BF), angle.sin().to(BF)
    kc, vc = (torch.zeros(batch, T, G, D, dtype=BF, device=cuda) for _ in range(2))
    k1, v1 = torch.zeros_like(kc), torch.zeros_like(vc)
    q = ops.qkv_rope_append(x, wqkv, nw, 1e-5, H, G, D, cos, sin, pos, kc, vc, seq_len=seq)
    each = [ops.qkv_rope_append(x[b * seq:(b + 1) * seq][:16], wqkv, nw, 1e-5, H, G, D, cos, sin, pos, k1[b:b + 1], v1[b:b + 1],
                                seq_len=min(seq, 16)) for b in range(batch)]
    for got, want in ((q.view(batch, seq, -1)[:, :16], torch.stack(each)), (kc[:, :pos + 16], k1[:, :pos + 16]), (vc[:, :pos + 16], v1[:, :pos + 16])):
        # two bf16 roundings (the projection's and the rotation's) and a normed value that rounds to its neighbour, of values up to 8
        assert (got.float() - want.float()).abs().max() <= 8 * 2.0 ** -7 and (got != want).float().mean() <= 0.1
    assert (kc[:, pos + seq:] == 0).all() and (kc[:, :pos] == 0).all()
