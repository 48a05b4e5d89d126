"""The tiled GEMM over its six tiles: edges of tiles, ragged rows, strips and K, row strides and row starts of any alignment,
against the product of the same bf16 values in 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _bound(x, w, y):
    """One rounding to bf16 of the result and K roundings to fp32 of partial sums."""
    return y.abs() * 2.0 ** -8 + x.shape[1] * 2.0 ** -24 * (x.abs() @ w.abs().t()) + 1e-30


# (rows, columns, K): the comment names the tile that the rule picks
SHAPES = [
    (65, 16, 8), (97, 40, 72), (320, 768, 768), (129, 1000, 520), (257, 2048, 2056),  # 32 x 32; K below, at and past a step
    (96, 6144, 768), (700, 1504, 1000), (193, 4100, 768),                             # 64 x 64
    (320, 6144, 712),                                                                 # 64 x 128
    (1000, 3096, 2008), (1030, 6104, 264),                                            # 128 x 128
    (2049, 2304, 768), (700, 6160, 776), (2100, 11264, 520),                          # 128 x 192
    (700, 17928, 1032),                                                               # 256 x 256
]


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
