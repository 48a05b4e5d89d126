"""LayerNorm whose rows stay in registers, at the widths where a thread's share of a row changes, against 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("rows,d", [(3, 8), (1, 2040), (5, 2048), (2, 2056), (300, 2560), (4, 4096), (3, 4104), (2, 8192), (2, 8200), (700, 768)])
def test_widths(cuda, rows, d):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(rows + d)
    x0 = (torch.randn(rows, d, generator=g, device=cuda) * 3 + 1).to(BF)
    w, b = (torch.randn(d, generator=g, device=cuda).to(BF) for _ in range(2))
    out = torch.full((rows + 1, d), 7.0, dtype=BF, device=cuda)
    got = ops.layernorm(x0, w, b, 1e-5, out=out[:rows])
    x = x0.double()
    mean = x.mean(-1, keepdim=True)
    n = (x - mean) / (((x - mean) ** 2).mean(-1, keepdim=True) + 1e-5).sqrt()
    want = n * w.double() + b.double()
    # one rounding of the result; sums of d terms in fp32 for the mean and the variance, of which a thread adds at most d / 256 + 8 in a row
    eps = (d / 256 + 16) * 2.0 ** -23
    bound = want.abs() * 2.0 ** -8 + (x.abs().mean(-1, keepdim=True) / x.std(-1, keepdim=True, unbiased=False) + n.abs()) * w.double().abs() * eps + 1e-6
    assert ((got.double() - want).abs() <= bound).all() and (out[rows] == 7.0).all()
