"""The norm of rows held by one wave against the one that takes rows of any start: the same bits, and against 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("d", [8, 248, 256, 264, 512, 520, 768, 1024, 1032, 2048, 2056, 4096, 4104, 36])
@pytest.mark.parametrize("rows", [1, 65, 1023, 1025])
def test_rows_of_one_wave(cuda, rows, d):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(rows + d)
    x = (torch.randn(rows, d, generator=g, device=cuda) * torch.logspace(-3, 3, rows, device=cuda)[:, None]).to(BF)
    w = (1 + 0.3 * torch.randn(d, generator=g, device=cuda)).to(BF)
    got = ops.rmsnorm(x, w)
    # a start that is not on 16 bytes takes the kernel of one workgroup per row
    flat = torch.empty(rows * d + 8, dtype=BF, device=cuda)
    odd = flat[1:1 + rows * d].view(rows, d)
    odd.copy_(x)
    assert torch.equal(got, ops.rmsnorm(odd, w))
    # two roundings to bf16 (2^-8 each), and the fp32 sum of d squares
    want = x.double() * (x.double().square().mean(-1, keepdim=True) + 1e-5).rsqrt() * w.double()
    assert ((got.double() - want).abs() <= want.abs() * (2.0 ** -7 + 2.0 ** -16 + d * 2.0 ** -24) + 1e-30).all()
    assert torch.equal(ops.rmsnorm(x, w, out=x), got)  # in place
