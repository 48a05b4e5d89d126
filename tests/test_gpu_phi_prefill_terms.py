"""Phi's attention over many new tokens in three-term bf16 products: every number of chunks with rotated features, queries that see infinities and queries
that do not, against 64 bits over the positions that a query sees."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _turn(x, cos, sin, half, rot):  # (n, H, D), a row of the tables each
    c, s, x = cos.double()[:, None], sin.double()[:, None], x.double()
    a, b, rest = x[..., :half], x[..., half:rot], x[..., rot:]
    return torch.cat([a * c - b * s, a * s + b * c, rest], -1)


def _case(cuda, B, S, H, D, rot, pos):
    g = torch.Generator(device=cuda).manual_seed(S + D + rot)
    T = pos + S
    q = (torch.randn(B, S, H, D, generator=g, device=cuda) * 2).to(BF)
    k, v = (torch.randn(B, T, H, D, generator=g, device=cuda).to(BF) for _ in range(2))
    ang = torch.rand(T, rot // 2, generator=g, device=cuda) * 6.28
    return q, k, v, ang.cos(), ang.sin()


def _plain(q, k, v, cos, sin, rot, pos):
    """(weighted sums, of the absolute values) of one sequence, a query's positions alone"""
    S, H, D = q.shape
    qt, kt = _turn(q, cos[pos:pos + S], sin[pos:pos + S], rot // 2, rot), _turn(k, cos, sin, rot // 2, rot)
    out, mass = (torch.empty(S, H, D, dtype=torch.float64, device=q.device) for _ in range(2))
    for s in range(S):
        n = pos + s + 1
        p = torch.softmax((qt[s][None] * kt[:n]).sum(-1) / D ** 0.5, 0)[..., None]
        out[s], mass[s] = (p * v[:n].double()).sum(0), (p * v[:n].double().abs()).sum(0)
    return out, mass


@pytest.mark.parametrize("D,rot", [(32, 32), (64, 48), (80, 16), (80, 48), (128, 32), (128, 96), (128, 128)])
@pytest.mark.parametrize("B,S,H,pos", [(1, 66, 2, 0), (2, 33, 9, 95), (1, 129, 3, 1)])
def test_every_number_of_chunks(cuda, B, S, H, pos, D, rot):
    from ohara_amd import ops

    q, k, v, cos, sin = _case(cuda, B, S, H, D, rot, pos)
    got = ops.phi_attn(q.view(B * S, H * D), k, v, cos, sin, rot, B, S, H, D, pos).view(B, S, H, D)
    for b in range(B):
        want, mass = _plain(q[b], k[b], v[b], cos, sin, rot, pos)
        # one rounding to bf16; scores are fp32 sums of D products that are 64 together at most, which their weights follow
        assert ((got[b].double() - want).abs() <= want.abs() * 2.0 ** -8 + mass * (D * 2.0 ** -18) + 1e-30).all()


@pytest.mark.parametrize("D,rot", [(32, 16), (64, 64), (80, 32), (128, 96), (128, 128)])
@pytest.mark.parametrize("B,S,H,pos,teams", [(1, 193, 3, 0, 2), (1, 257, 2, 0, 2), (2, 16, 5, 240, 2), (1, 70, 3, 187, 2), (1, 130, 9, 380, 2), (1, 600, 32, 0, 2), (4, 200, 17, 0, 1),
                                             (1, 192, 3, 0, 1)])
def test_two_teams(cuda, B, S, H, pos, teams, D, rot):
    """The last round with a tile for one team and for both, waves that see nothing of the second one's, on either side of the rule."""
    from ohara_amd import ops
    from ohara_amd._lib import lib

    assert lib().ohara_phi_prefill_teams(B, S, H, pos) == teams
    q, k, v, cos, sin = _case(cuda, B, S, H, D, rot, pos)
    got = ops.phi_attn(q.view(B * S, H * D), k, v, cos, sin, rot, B, S, H, D, pos).view(B, S, H, D)
    b = B - 1
    want, mass = _plain(q[b], k[b], v[b], cos, sin, rot, pos)
    assert ((got[b].double() - want).abs() <= want.abs() * 2.0 ** -8 + mass * (D * 2.0 ** -18) + 1e-30).all()


@pytest.mark.parametrize("D,rot", [(16, 16), (32, 32), (64, 48), (80, 16), (80, 48), (128, 32), (128, 96), (128, 128)])
@pytest.mark.parametrize("B,S,H,teams", [(1, 257, 5, 2), (4, 200, 17, 1)])
def test_three_terms(cuda, B, S, H, teams, D, rot):
    """Few outputs are another bf16 number than the rounded one of 64 bits: 0.00 to 0.04 % where all the terms are in the sums, 0.3 % and more where the third
    ones of a product are not, which the bounds above would let pass."""
    from ohara_amd import ops
    from ohara_amd._lib import lib

    assert lib().ohara_phi_prefill_teams(B, S, H, 0) == teams
    q, k, v, cos, sin = _case(cuda, B, S, H, D, rot, 0)
    got = ops.phi_attn(q.view(B * S, H * D), k, v, cos, sin, rot, B, S, H, D, 0).view(B, S, H, D)
    want, _ = _plain(q[B - 1], k[B - 1], v[B - 1], cos, sin, rot, 0)
    assert want.numel() > 20000 and (got[B - 1] != want.to(BF)).sum() <= want.numel() // 1000


@pytest.mark.parametrize("S,at", [(100, 0), (100, 20), (100, 63), (100, 64), (100, 99), (200, 63), (200, 64), (200, 130), (200, 199)])
def test_infinities(cuda, S, at):
    """A key of minus infinity in a feature that is not rotated has no weight, one in a rotated feature may have none; an infinite value reaches the
    queries that see it."""
    from ohara_amd import ops

    H, D, rot = 3, 80, 32
    for what in ("plain key", "rotated key", "value"):
        q, k, v, cos, sin = _case(cuda, 1, S, H, D, rot, 0)
        q, k = q.abs() + 0.25, k.clone()
        if what == "value":
            v[0, at, 1, 7] = float("inf")
        else:
            k[0, at, 1, 40 if what == "plain key" else 3] = float("-inf")
        got = ops.phi_attn(q.view(S, H * D), k, v, cos, sin, rot, 1, S, H, D, 0).view(S, H, D).double()
        want, mass = _plain(q[0], k[0], v[0], cos, sin, rot, 0)
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got.isinf(), want.isinf())
        ok = want.isfinite()
        assert ok.any()
        bound = want.abs() * 2.0 ** -8 + mass * (D * 2.0 ** -18) + 1e-30
        assert ((got - want).abs()[ok] <= bound[ok]).all()
