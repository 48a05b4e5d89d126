"""Products with a residual and the norm behind them in two parts of a depth under 2048, at the rows where they begin and end and where tiles do, against 64 bits and the product
over the whole depth."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

# columns, depth, rows, parts
SHAPES = [
    (768, 768, 32, 1), (768, 768, 33, 2), (768, 768, 65, 2), (768, 768, 128, 2), (768, 768, 159, 2), (768, 768, 700, 1), (640, 768, 97, 2), (512, 1024, 97, 1), (768, 640, 100, 1),
    (512, 768, 97, 1), (512, 1280, 33, 2), (512, 1280, 190, 2), (512, 1792, 250, 2), (384, 1280, 97, 2), (256, 1536, 500, 2), (16, 1024, 130, 1),
    (1024, 1024, 70, 2), (1536, 1536, 190, 2), (640, 1536, 300, 2), (768, 1792, 193, 2),
]


@pytest.mark.parametrize("n,k,rows,parts", SHAPES)
def test_residual_and_norm(cuda, n, k, rows, parts):
    from ohara_amd import ops
    from ohara_amd._lib import check, lib

    g = torch.Generator(device=cuda).manual_seed(n + k + rows)
    x, w, res = (torch.randn(*s, generator=g, device=cuda).to(BF) for s in ((rows, k), (n, k), (rows, n)))
    norm = torch.randn(n, generator=g, device=cuda).to(BF)
    room = lib().ohara_gemm_residual_norm_bytes(rows, n, k)
    assert room == (0 if parts == 1 else parts * rows * n * 4)
    packed = ops.pack_linear(w)
    xd, wd = x.double(), w.double()
    y = xd @ wd.t()
    # k roundings to fp32 of partial sums, one of the product to bf16 and one of the sum with the residual
    bound = (xd.abs() @ wd.abs().t()) * k * 2.0 ** -24 + y.abs() * 2.0 ** -8
    bound = bound * 1.01 + (y + res.double()).abs() * 2.0 ** -8 + bound * 2.0 ** -8
    for given in {room, 0}:
        ws = torch.empty(max(given, 1), dtype=torch.uint8, device=cuda)
        out, xn = res.clone(), torch.full((rows + 1, n), 7.0, dtype=BF, device=cuda)
        check(lib().ohara_gemm_residual_norm_bf16(x.data_ptr(), k, packed.data.data_ptr(), n, k, rows, out.data_ptr(), norm.data_ptr(), 1e-5,
                                                  xn.data_ptr(), ws.data_ptr(), given, torch.cuda.current_stream().cuda_stream), "residual_norm")
        assert ((out.double() - (y + res.double())).abs() <= bound).all()
        assert torch.equal(xn[:rows], ops.rmsnorm(out, norm, 1e-5)) and (xn[rows] == 7.0).all()
