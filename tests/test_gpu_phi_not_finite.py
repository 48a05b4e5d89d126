"""Phi's attention of one token over keys that are not numbers or minus infinity: a NaN reaches its row also where no other position is in its group of
lanes, its team or its chunk, and minus infinity has no weight also where it comes first."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

# (position of the key, of the query): a group's only one, a chunk's first of several, a chunk's only one, the one of a third chunk, a four's only one
PLACES = [(3, 5), (70, 80), (0, 100), (64, 64), (128, 128), (256, 256), (17, 300)]


def _setup(cuda, B, H, D, rot):
    from ohara_amd.phi import rope_cos_sin

    g = torch.Generator(device=cuda).manual_seed(H + D)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda).to(BF)  # noqa: E731
    return r, r(B, H * D).abs() + 0.25, r(B, 512, H, D), r(B, 512, H, D), *(t.to(cuda) for t in rope_cos_sin(512, rot))


def _plain(q, k, v, cos, sin, rot, pos):
    """In 64 bits, and a bound: scores are fp32 sums of D products, which their weights follow (a key of minus infinity has none)."""
    half, D = rot // 2, q.shape[-1]

    def turned(x, c, s):
        a, b, rest = x[..., :half], x[..., half:rot], x[..., rot:]
        return torch.cat([a * c - b * s, a * s + b * c, rest], -1)

    c, s = cos.double(), sin.double()
    qr, kr = turned(q.double(), c[pos], s[pos]), turned(k[:, :pos + 1].double(), c[:pos + 1, None], s[:pos + 1, None])
    p = torch.softmax((qr[:, None] * kr).sum(-1) * D ** -0.5, 1)[..., None]
    near = (qr[:, None].abs() * kr.abs().nan_to_num(0.0, 0.0, 0.0)).sum(-1).amax(1) * D ** -0.5
    vd = v[:, :pos + 1].double()
    want = (p * vd).sum(1)
    return want, want.abs() * 2.0 ** -8 + (p * vd.abs()).sum(1) * (near * (D + 4) * 2.0 ** -23 + 2.0 ** -18)[..., None] + 1e-30


def _holds(got, want, bound, what, at, pos):
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan), (what, at, pos)
    assert ((got.double() - want).abs() <= bound)[~nan].all(), (what, at, pos)


# batch, heads, head width, rotated, chunks, rows of the product beside it (0: none)
@pytest.mark.parametrize("B,H,D,rot,ns,n", [(1, 4, 64, 32, 1, 0), (2, 5, 80, 32, 1, 0), (1, 32, 80, 32, 16, 0), (3, 4, 40, 12, 4, 0), (40, 4, 128, 128, 1, 0),
                                            (1, 32, 80, 32, 16, 2560), (4, 24, 80, 32, 8, 1024)])
def test_one_token(cuda, B, H, D, rot, ns, n):
    from ohara_amd import ops

    r, q, keys, values, cos, sin = _setup(cuda, B, H, D, rot)
    ws = ops.phi_attn_workspace(B, H, D, ns, cuda) if ns > 1 else None
    x, bias, w = r(B, 10240), r(n), ops.pack_linear(r(n, 10240)) if n else None
    for at, pos in PLACES:
        for what in ("nan", "-inf")[:1 + (rot < D)]:
            bad = keys.clone()
            bad[0, at, 1, D - 1] = float(what)  # (not a rotated feature, but where all are)
            if n:
                got, _ = ops.phi_attn_linear(q, bad, values, cos, sin, rot, B, H, D, pos, x, w, bias, None, n_split=ns, workspace=ws)
            else:
                got = ops.phi_attn(q, bad, values, cos, sin, rot, B, 1, H, D, pos, n_split=ns, workspace=ws)
            want, bound = _plain(q.view(B, H, D), bad, values, cos, sin, rot, pos)
            assert (want[0, 1].isnan().all() if what == "nan" else want.isfinite().all()) and want[:, 0].isfinite().all()
            _holds(got.view(B, H, D), want, bound, what, at, pos)


@pytest.mark.parametrize("B,H,D,rot,ns,n,k", [(1, 32, 80, 32, 16, 2560, 10240), (2, 32, 80, 32, 8, 2560, 2560)])
def test_merged_by_the_projection(cuda, B, H, D, rot, ns, n, k):
    """The projection's weights are a unit matrix and its addends zero, so its output is the attention's."""
    from ohara_amd import ops

    r, q, keys, values, cos, sin = _setup(cuda, B, H, D, rot)
    ws = ops.phi_attn_workspace(B, H, D, ns, cuda)
    x, none, w = r(B, k), torch.zeros(n, dtype=BF, device=cuda), ops.pack_linear(torch.zeros(n, k, dtype=BF, device=cuda))
    unit, zero = ops.pack_linear(torch.eye(n, H * D, device=cuda).to(BF)), torch.zeros(B, n, dtype=BF, device=cuda)
    y, out = torch.empty_like(zero), torch.empty_like(zero)
    reached = [p for p in PLACES if ops.phi_attn_out_chunks(B, H, D, rot, ns, p[1], n, k)]
    assert len(reached) >= 4
    for at, pos in reached:
        for what in ("nan", "-inf"):
            bad = keys.clone()
            bad[0, at, 1, D - 1] = float(what)
            ws[-ws.numel() // 2:] = 255  # (not numbers: sums of chunks that this call does not have)
            ops.phi_attn_out(q, bad, values, cos, sin, rot, B, H, D, pos, x, w, none, None, y, ns, ws, unit, none, zero, out)
            if what == "nan":  # (a row of the product: in every column)
                assert out[0].isnan().all() and (B == 1 or out[1].isfinite().all()), (at, pos)
            else:
                want, bound = _plain(q.view(B, H, D), bad, values, cos, sin, rot, pos)
                _holds(out.view(B, H, D), want, bound, what, at, pos)


# (two sequences of one team of waves, one of two)
@pytest.mark.parametrize("B,S,H,pos", [(2, 70, 9, 20), (1, 193, 3, 0)])
@pytest.mark.parametrize("D,rot", [(16, 16), (32, 16), (64, 64), (80, 48), (128, 32), (128, 128)])
def test_prompts(cuda, B, S, H, pos, D, rot):
    """Queries that see something that is not finite are walked again, the others are not; each has its own positions' sums."""
    from test_gpu_phi_prefill_terms import _case, _plain as plain

    from ohara_amd import ops

    q, k, v, cos, sin = _case(cuda, B, S, H, D, rot, pos)
    q, T = q.abs() + 0.25, pos + S
    for at in (0, 15, pos + 16, pos + 63, T - 1):
        for what in ("nan", "rotated key", "plain key", "value"):
            bad, worse = k.clone(), v.clone()
            if what == "value":
                worse[B - 1, at, 1, D - 3] = float("inf")
            elif what == "plain key" and rot < D:
                bad[B - 1, at, 1, D - 1] = float("-inf")
            else:
                bad[B - 1, at, 1, 3] = float("nan" if what == "nan" else "-inf")
            got = ops.phi_attn(q.view(B * S, H * D), bad, worse, cos, sin, rot, B, S, H, D, pos).view(B, S, H, D)[B - 1].double()
            want, mass = plain(q[B - 1], bad[B - 1], worse[B - 1], cos, sin, rot, pos)
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf()), (at, what)
            ok = want.isfinite()
            assert ok.any() and ((got - want).abs() <= want.abs() * 2.0 ** -8 + mass * (D * 2.0 ** -18) + 1e-30)[ok].all(), (at, what)


def test_prompts_are_not_held_up(cuda):
    """A NaN in every head's first key, so that all queries are walked again: a quarter of the time that they take one by one, a position at a time, which is
    240 to 280 times the finite call's."""
    from ohara_amd import ops
    from ohara_amd.phi import rope_cos_sin

    S, H, D, rot = 700, 32, 80, 32
    q, k, v = (torch.randn(1, S, H, D, device=cuda).to(BF) for _ in range(3))
    cos, sin = (t.to(cuda) for t in rope_cos_sin(S, rot))

    def least(n):
        times = []
        for _ in range(n):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            ops.phi_attn(q.view(S, H * D), k, v, cos, sin, rot, 1, S, H, D, 0)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    finite = least(10)
    k[0, 0] = float("nan")
    assert least(5) <= 60 * finite
