"""The projection of up to 64 rows onto many columns (a vocabulary), where every workgroup norms all rows: edges of K, of rows and of columns,
against the norm and the projection as two calls."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("n,k", [(16384, 8), (16400, 512), (16392, 520), (32768, 768), (17000, 1024), (16389, 1032), (16400, 1544), (16384, 2048), (16400, 2056)])
@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17, 32, 33, 48, 64])
def test_store(cuda, rows, n, k):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(rows + n + k)
    x = (torch.randn(rows, k, generator=g, device=cuda) * torch.logspace(-2, 2, rows, device=cuda)[:, None]).to(BF)
    nw = (1 + 0.3 * torch.randn(k, generator=g, device=cuda)).to(BF)
    w = (torch.randn(n, k, generator=g, device=cuda) * 0.05).to(BF)
    packed, xn = ops.pack_linear(w), ops.rmsnorm(x, nw, 1e-5)
    # the normed rows may round to a neighbour (2^-8 of a value at most: the sum of squares is in another order), results by 2^-8, sums by K 2^-24
    for got, rows_in in ((ops.gemm_skinny(x, packed, nw, 1e-5), xn), (ops.gemm_skinny(xn, packed), xn)):
        ref, mass = rows_in.double() @ w.double().t(), rows_in.double().abs() @ w.double().abs().t()
        assert ((got.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + mass * (2.0 ** -8 + k * 2.0 ** -24)).all()
    plain = ops.gemm_skinny(xn, packed).double()
    assert ((plain - ref).abs() <= ref.abs() * 2.0 ** -8 + mass * k * 2.0 ** -24).all()
    assert (ops.gemm_skinny(x, packed, nw, 1e-5).double() != plain).float().mean() <= 0.05
