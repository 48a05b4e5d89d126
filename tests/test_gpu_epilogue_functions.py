"""The epilogues' silu and gelu over every bf16 number."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _every(cuda):
    return torch.arange(65536, device=cuda, dtype=torch.int32).to(torch.int16).view(BF)


@pytest.mark.parametrize("rows", [1, 65, 300])
def test_gelu(cuda, rows):
    """Of a bias alone, op by op as the reference's bf16 path (phi.py:37-40)."""
    from ohara_amd import ops

    x = _every(cuda)
    w = ops.pack_linear(torch.zeros(65536, 8, dtype=BF, device=cuda))
    got = ops.linear_bias(torch.ones(rows, 8, dtype=BF, device=cuda), w, x, "gelu")
    cube = x * x * x
    inner = (0.7978845608028654 * (x + (0.044715 * cube).to(BF)).to(BF).float()).to(BF)
    want = (0.5 * x).to(BF).float() * (1.0 + torch.tanh(inner.float()).to(BF).float()).to(BF).float()
    assert torch.allclose(got.float(), want.to(BF).float().expand(rows, -1), rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("rows,n", [(65, 65536), (8192, 6144)])
def test_silu(cuda, rows, n):
    """Of weights times a one, the other factor one: the small tiles, the large ones, and numbers below -87 among the others and not."""
    from ohara_amd import ops

    for x in (_every(cuda), _every(cuda).clamp(min=-87).nan_to_num(1.0)):
        x = x[torch.randperm(65536, device=cuda)[:n]] if n < 65536 else x
        gate, up = torch.zeros(n, 64, dtype=BF, device=cuda), torch.zeros(n, 64, dtype=BF, device=cuda)
        gate[:, 3], up[:, 3] = x, 1.0
        row = torch.zeros(rows, 64, dtype=BF, device=cuda)
        row[:, 3] = 1.0
        got = ops.gemm(row, ops.pack_gate_up(gate, up))
        d = x.double()
        want = (d / (1.0 + torch.exp(-d))).to(BF)
        plain = d.isfinite() & (d >= -87)  # (below: a reciprocal beyond fp32's normal numbers; infinities times the other columns' zeros are NaN)
        assert torch.equal(got[:, plain], want[plain].expand(rows, -1))
        small = d.isfinite() & (d < -87)
        assert (got[:, small].abs() <= 1e-35).all()
