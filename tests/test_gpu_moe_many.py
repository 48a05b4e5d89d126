"""The sort and the experts over many (token, expert) pairs: both tiles, experts with no, one, a tile's and a tile and one
pairs, against plain sorts and products in 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _sort(idx, E, cuda):
    from ohara_amd._lib import check, lib

    n = idx.numel()
    offs, pair_of, pos_of = (torch.full((m,), -1, dtype=torch.int32, device=cuda) for m in (E + 1, n, n))
    check(lib().ohara_moe_sort_pairs(idx.data_ptr(), n, E, offs.data_ptr(), pair_of.data_ptr(), pos_of.data_ptr(),
                                     torch.cuda.current_stream().cuda_stream), "sort")
    return offs, pair_of, pos_of


@pytest.mark.parametrize("pairs,experts", [(1025, 64), (1024, 65), (2049, 3), (5000, 1), (30720, 64), (65536, 1024), (4097, 1000)])
def test_sort_of_many_pairs_is_stable(cuda, pairs, experts):
    g = torch.Generator().manual_seed(pairs + experts)
    idx = torch.randint(0, experts, (pairs,), generator=g, dtype=torch.int32)
    idx[pairs // 3: pairs // 2] = experts // 2  # one expert has a run to itself
    offs, pair_of, pos_of = _sort(idx.to(cuda), experts, cuda)
    order = torch.argsort(idx.long(), stable=True)
    assert torch.equal(pair_of.cpu().long(), order)
    assert offs[0] == 0 and torch.equal(offs.cpu().long()[1:], torch.bincount(idx.long(), minlength=experts).cumsum(0))
    assert torch.equal(pos_of.cpu().long()[order], torch.arange(pairs))


# pairs per expert: streams of 16, tiles of 64 and 128; widths off a strip; K off a step
@pytest.mark.parametrize("counts,d,hidden,top", [
    ([3, 0, 1, 9], 72, 24, 1), ([64, 0, 1, 33, 100, 66], 136, 40, 2), ([65, 64, 0, 130, 255, 1, 200, 69], 264, 88, 4),
    ([20, 64, 65, 0, 1], 520, 264, 2),
    ([500, 0, 129, 128, 1, 400], 1024, 512, 1), ([256, 258], 520, 96, 2),
    ([20, 33, 0, 40, 64, 1], 1024, 512, 1), ([30, 17, 65, 0], 64, 128, 2),  # tiles of 64, K of whole steps: many, one, two
])
def test_experts_over_many_pairs(cuda, counts, d, hidden, top):
    from ohara_amd import ops
    from ohara_amd._lib import check, lib

    E, pairs = len(counts), sum(counts)
    assert pairs % top == 0
    g = torch.Generator(device=cuda).manual_seed(pairs + d)
    x = torch.randn(pairs // top, d, generator=g, device=cuda).to(BF)
    gate, up = ((torch.randn(E, hidden, d, generator=g, device=cuda) * d ** -0.5).to(BF) for _ in range(2))
    down = (torch.randn(E, d, hidden, generator=g, device=cuda) * hidden ** -0.5).to(BF)
    wt = torch.rand(pairs, generator=g, device=cuda).to(BF)
    perm = ops.swiglu_perm(hidden, cuda)
    gu = torch.stack([ops.pack_rows(torch.cat([gate[e], up[e]]).contiguous(), perm, perm.numel()) for e in range(E)]).contiguous()
    dn = torch.stack([ops.pack_rows(down[e].contiguous()) for e in range(E)]).contiguous()
    idx = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(pairs, generator=torch.Generator().manual_seed(1))]
    offs, pair_of, _ = _sort(idx.to(cuda, torch.int32), E, cuda)
    act = torch.full((pairs, hidden), float("nan"), device=cuda, dtype=BF)
    y = torch.full((pairs, d), float("nan"), device=cuda, dtype=BF)
    st = torch.cuda.current_stream().cuda_stream
    check(lib().ohara_moe_experts_gate_up_many(x.data_ptr(), d, gu.data_ptr(), gu.stride(0) * 2, E, hidden, d, top, pairs,
                                               offs.data_ptr(), pair_of.data_ptr(), act.data_ptr(), hidden, st), "gate_up")
    check(lib().ohara_moe_experts_down_many(act.data_ptr(), hidden, dn.data_ptr(), dn.stride(0) * 2, E, d, hidden, top, pairs,
                                            offs.data_ptr(), pair_of.data_ptr(), wt.data_ptr(), y.data_ptr(), d, st), "down")
    eps = 2.0 ** -8
    for e, n in enumerate(counts):
        at = pair_of[offs[e]: offs[e + 1]].long()
        if not n:
            continue
        rows, a, out = x[at // top].double(), act[offs[e]: offs[e + 1]].double(), y[offs[e]: offs[e + 1]].double()
        gv, uv = rows @ gate[e].double().t(), rows @ up[e].double().t()
        # gate and up are rounded to bf16, so is silu (whose slope is below 1.1), so is the product; K roundings of fp32 sums
        slack = d * 2.0 ** -24 * d ** 0.5
        want = gv * gv.sigmoid() * uv
        bound = eps * (1.1 * gv.abs() * uv.abs() + 3 * want.abs()) + slack * (gv.abs() + uv.abs() + 1) + 1e-30
        assert ((a - want).abs() <= bound).all()
        yv = a @ down[e].double().t()
        want = yv * wt[at].double()[:, None]
        assert ((out - want).abs() <= 2 * eps * want.abs() + hidden * 2.0 ** -24 * (a.abs() @ down[e].double().abs().t()) + 1e-30).all()
