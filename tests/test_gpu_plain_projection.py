"""Projections of up to 64 rows without a norm, where a wave requests its whole share of K at once: every share, K at its edges, whole
strips and halves, rows at the edges of a block, plain and with a residual, against 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("k", [8, 24, 264, 768, 1000, 1024, 1032, 1288, 1544, 1800, 2048, 2064, 2312, 2568, 2824, 3072, 3080, 3584, 4096, 4104, 4616, 5128, 5632, 5640, 6144, 6152])
@pytest.mark.parametrize("n", [40, 771, 2064, 4104])
def test_plain_projection(cuda, n, k):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(n + k)
    w = (torch.randn(n, k, generator=g, device=cuda) * 0.05).to(BF)
    packed, w64 = ops.pack_linear(w), w.double()
    for rows in (1, 7, 8, 16, 17, 33, 64):
        x = torch.randn(rows, k, generator=g, device=cuda).to(BF)
        want, mass = x.double() @ w64.t(), x.double().abs() @ w64.abs().t()
        bound = want.abs() * 2.0 ** -8 + mass * k * 2.0 ** -24
        assert ((ops.gemm_skinny(x, packed).double() - want).abs() <= bound).all()
        r = torch.randn(rows, n, generator=g, device=cuda).to(BF)
        # the sum with the residual is of the rounded product, and rounded itself
        both = (r.double() + want).abs() * 2.0 ** -8 + bound * (1 + 2.0 ** -8)
        assert ((ops.gemm_skinny(x, packed, residual=r).double() - (r.double() + want)).abs() <= both).all()
