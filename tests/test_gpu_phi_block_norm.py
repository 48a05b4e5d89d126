"""Phi's block head on one or two rows before their LayerNorm: the bits of the norm's own launch and the head behind it, over widths that end inside a
k-step, strips that end inside sixteen columns, and as many of them as workgroups, more, and twice as many."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("B,S", [(1, 1), (2, 1), (1, 2)])
@pytest.mark.parametrize("d,ff", [(2048, 260), (2048, 8192), (2064, 2000), (2320, 12), (2560, 10240), (2560, 8708)])
def test_the_norm_inside(cuda, B, S, d, ff):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(d + ff + B)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda)  # noqa: E731
    rows, H, D, T, pos = B * S, d // 16, 16, 8, 3
    assert ops.phi_block_norms(rows, d, ff)
    x, lw, lb, b = (2 * r(rows, d) + 1).to(BF), (1 + r(d) / 8).to(BF), r(d).to(BF), r(3 * d + ff).to(BF)
    w = ops.pack_linear((r(3 * d + ff, d) / 16).to(BF))

    def outs():
        return [torch.full(s, 7.0, dtype=BF, device=cuda) for s in ((B, T, H, D), (B, T, H, D), (rows, d), (rows, ff))]

    want, got, replayed = outs(), outs(), outs()
    ops.phi_block_in(ops.layernorm(x, lw, lb), None, None, 1e-5, w, b, d, ff, B, S, pos, *want)
    ops.phi_block_in(x, lw, lb, 1e-5, w, b, d, ff, B, S, pos, *got)
    graph = torch.cuda.CUDAGraph()
    dev = torch.zeros(1, dtype=torch.int32, device=cuda) if S == 1 else None
    with torch.cuda.graph(graph):
        ops.phi_block_in(x, lw, lb, 1e-5, w, b, d, ff, B, S, pos, *replayed, dev)
    if dev is not None:
        dev.fill_(pos)
    graph.replay()
    for a, one, two in zip(want, got, replayed):
        assert torch.equal(a, one) and torch.equal(a, two)


def test_elsewhere_a_launch_of_its_own(cuda):
    from ohara_amd import ops

    for no in ((3, 2560, 10240), (1, 2576, 10240), (1, 2032, 8192), (1, 2048, 240), (0, 2560, 10240), (1, 2560, 0)):
        assert not ops.phi_block_norms(*no)
