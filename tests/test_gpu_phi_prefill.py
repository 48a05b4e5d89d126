"""Phi's attention over many new tokens at every head width it takes: rotated features in eights and not, tables that start off 16 bytes,
edges of tiles and of the workgroup's queries, positions before them, against 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("D,rot", [(16, 16), (32, 16), (64, 32), (64, 20), (80, 32), (80, 80), (128, 64), (128, 12)])
@pytest.mark.parametrize("B,S,H,pos", [(1, 16, 3, 0), (2, 65, 8, 31), (1, 200, 5, 33), (3, 97, 16, 0), (1, 64, 1, 190)])
@pytest.mark.parametrize("start", [0, 1])
def test_against_64_bits(cuda, B, S, H, pos, D, rot, start):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(S + D + rot)
    T, half = pos + S + 2, rot // 2
    q = (torch.randn(B, S, H, D, generator=g, device=cuda) * 2).to(BF)
    k, v = (torch.randn(B, T, H, D, generator=g, device=cuda).to(BF) for _ in range(2))
    ang = torch.rand(T, half, generator=g, device=cuda) * 6.28
    cos, sin = (torch.cat([torch.zeros(start, device=cuda), t.reshape(-1)])[start:].view(T, half) for t in (ang.cos(), ang.sin()))

    def turn(x, at):  # (B, n, H, D) at positions `at`
        c, s = (t.double()[at][None, :, None] for t in (cos, sin))
        x = x.double()
        a, b, rest = x[..., :half], x[..., half:rot], x[..., rot:]
        return torch.cat([a * c - b * s, a * s + b * c, rest], -1)

    at = torch.arange(T, device=cuda)
    qt, kt = turn(q, at[pos:pos + S]), turn(k[:, :pos + S], at[:pos + S])
    score = torch.matmul(qt.transpose(1, 2), kt.permute(0, 2, 3, 1).contiguous()) / D ** 0.5
    score.masked_fill_(at[None, :pos + S] > at[pos:pos + S, None], float("-inf"))
    p, vt = torch.softmax(score, -1), v[:, :pos + S].double().transpose(1, 2).contiguous()
    want, mass = (torch.matmul(p, t).transpose(1, 2) for t in (vt, vt.abs()))
    k[:, pos + S:] = float("nan")
    v[:, pos + S:] = float("nan")
    got = ops.phi_attn(q.view(B * S, H * D), k, v, cos, sin, rot, B, S, H, D, pos).view(B, S, H, D)
    # one rounding to bf16; scores are fp32 sums of D products that are 64 together at most, which their weights follow
    assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + mass * (D * 2.0 ** -18) + 1e-30).all()
