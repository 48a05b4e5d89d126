"""Phi's attention of one token with a product beside it: the product's bits are those of a launch of its own, the attention against 64 bits, over chunks
that begin, fill and end, replayed from a graph with other positions, and where the two go out by themselves."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _attention(q, k, v, cos, sin, rot, pos):
    """In 64 bits, with the bound: an fp32 sum of D products a score (which its weight follows), of the positions' values, and one rounding."""
    D, half = q.shape[-1], rot // 2

    def turned(x, c, s):
        a, b, rest = x[..., :half], x[..., half:rot], x[..., rot:]
        return torch.cat([a * c - b * s, a * s + b * c, rest], -1)

    c, s = cos.double(), sin.double()
    qr = turned(q.double(), c[pos], s[pos])  # (B, H, D)
    kr = turned(k[:, :pos + 1].double(), c[:pos + 1, None], s[:pos + 1, None])  # (B, T, H, D)
    sc = (qr[:, None] * kr).sum(-1) * D ** -0.5
    near = (qr[:, None].abs() * kr.abs()).sum(-1).amax(1) * D ** -0.5
    p = torch.softmax(sc, 1)[..., None]
    vd = v[:, :pos + 1].double()
    want = (p * vd).sum(1)
    return want, want.abs() * 2.0 ** -8 + (p * vd.abs()).sum(1) * (near * (D + 4) * 2.0 ** -23 + 2.0 ** -18)[..., None] + 1e-30


# batch, heads, head width, rotated, chunks, rows and depth of the product (the first four: one launch at all positions; the last five: two launches)
SHAPES = [
    (1, 3, 128, 16, 64, 2560, 10240), (2, 16, 64, 64, 16, 3000, 10240), (4, 24, 80, 32, 8, 1024, 10240),
    (1, 32, 80, 32, 16, 2560, 10240), (1, 32, 80, 32, 5, 2556, 2048), (2, 16, 64, 64, 16, 40, 2056), (1, 3, 128, 16, 64, 1000, 2304),
    (1, 32, 80, 32, 1, 2560, 2048), (4, 24, 80, 32, 8, 16, 2048),
    (2, 32, 80, 32, 8, 2560, 2304), (1, 8, 24, 12, 4, 64, 2048), (1, 8, 64, 32, 4, 64, 264), (17, 2, 64, 32, 4, 64, 2048),
    (16, 32, 80, 40, 1, 16, 2048),
]


@pytest.mark.parametrize("B,H,D,rot,ns,n,k", SHAPES)
def test_beside_a_product(cuda, B, H, D, rot, ns, n, k):
    from ohara_amd import ops
    from ohara_amd.phi import rope_cos_sin

    T = 2048
    g = torch.Generator(device=cuda).manual_seed(H + D + ns + n)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda).to(BF)  # noqa: E731
    q, keys, values, x, bias, w = r(B, H * D), r(B, T, H, D), r(B, T, H, D), r(B, k), r(n), ops.pack_linear(r(n, k))
    cos, sin = (t.to(cuda) for t in rope_cos_sin(T, rot))
    ws = ops.phi_attn_workspace(B, H, D, ns, cuda) if ns > 1 else None
    alone = ops.linear_bias(x, w, bias)
    out, y, dev = torch.empty(B, H * D, dtype=BF, device=cuda), torch.empty(B, n, dtype=BF, device=cuda), torch.zeros(1, dtype=torch.int32, device=cuda)

    def call(pos, pos_dev):
        ops.phi_attn_linear(q, keys, values, cos, sin, rot, B, H, D, pos, x, w, bias, pos_dev, out=out, y=y, n_split=ns, workspace=ws)

    def check(pos):
        want, bound = _attention(q.view(B, H, D), keys, values, cos, sin, rot, pos)
        assert torch.equal(y, alone) and ((out.view(B, H, D).double() - want).abs() <= bound).all()
        out.fill_(7.0)
        y.fill_(7.0)

    places = [0, 1, 15, 16, 31, 63, 64, 65, 127, 128, 500, 64 * ns - 1, 64 * ns, 1749, 1750, 2047]
    places = sorted({p for p in places if p < T})
    if SHAPES.index((B, H, D, rot, ns, n, k)) < 4:
        from ohara_amd._lib import lib

        assert all(lib().ohara_phi_attn_linear_chunks(B, H, D, ns, p, n, k) > 0 for p in places)
    for pos in places:
        call(pos, None)
        check(pos)
        alone_out = ops.phi_attn(q, keys, values, cos, sin, rot, B, 1, H, D, pos, n_split=ns, workspace=ws)
        want, bound = _attention(q.view(B, H, D), keys, values, cos, sin, rot, pos)
        assert ((alone_out.view(B, H, D).double() - want).abs() <= bound).all()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(0, dev)
    for pos in places:
        dev.fill_(pos)
        graph.replay()
        check(pos)


def test_refused(cuda):
    from ohara_amd import ops
    from ohara_amd._lib import lib

    q, kv, w = torch.zeros(1, 64, dtype=BF, device=cuda), torch.zeros(1, 8, 1, 64, dtype=BF, device=cuda), torch.zeros(16, 2048, dtype=BF, device=cuda)
    x, bias, angles = torch.zeros(1, 2048, dtype=BF, device=cuda), torch.zeros(16, dtype=BF, device=cuda), torch.zeros(8, 16, device=cuda)
    packed = ops.pack_linear(w)
    out, y = torch.empty_like(q), torch.empty(1, 16, dtype=BF, device=cuda)

    def status(pos=0, ns=1, ldx=2048, n=16, wp=packed.data.data_ptr()):
        return lib().ohara_phi_attn_linear_bf16(q.data_ptr(), 64, kv.data_ptr(), kv.data_ptr(), angles.data_ptr(), angles.data_ptr(), 32, 1, 1, 64, 8, pos,
                                                None, ns, None, out.data_ptr(), x.data_ptr(), ldx, wp, n, 2048, bias.data_ptr(), y.data_ptr(), 16,
                                                torch.cuda.current_stream().cuda_stream)

    assert status() == 0
    assert all(s == -1 for s in (status(pos=8), status(ns=2), status(ldx=2040), status(ldx=2052), status(n=18), status(wp=None)))
    with pytest.raises(ValueError, match="weight is"):
        ops.phi_attn_linear(q, kv, kv, angles, angles, 32, 1, 1, 64, 0, x[:, :2040], packed, bias)


def _phi(cuda, **kw):
    from ohara_amd.phi import Phi, PhiConfig
    from oracle import phi_ref as P

    kw = dict(vocab_size=96, max_sequence_length=64, hidden_size=512, num_attention_heads=8, num_hidden_layers=2, rotary_dim=0.5, **kw)
    return Phi(PhiConfig(**kw), P.init_weights(P.RefPhiConfig(**kw), seed=2, dtype=BF), device=cuda)


@pytest.mark.parametrize("B", [1, 16, 17, 32, 33, 40])
def test_deep_product_of_many_sequences(cuda, monkeypatch, B):
    """One token each: the second product of the MLP goes beside the attention up to sixteen sequences; of more it takes the addends, as
    the product that 33 rows and more multiply in parts of the depth, and as the prompt's."""
    from ohara_amd import ops
    from ohara_amd._lib import lib

    m = _phi(cuda)
    assert lib().ohara_linear_bias_add2_bytes(33, 512, 2048) > 0
    g = torch.Generator(device=cuda).manual_seed(B)
    ids = torch.randint(0, 96, (B, 5), generator=g, device=cuda)
    cache = m.build_kv_cache(B)
    m(ids[:, :4], cache, 0)
    seen, linear_bias = [], ops.linear_bias

    def spy(x, w, bias, epilogue="bias", **kw):
        seen.append((w.k, epilogue))
        return linear_bias(x, w, bias, epilogue, **kw)

    monkeypatch.setattr(ops, "linear_bias", spy)
    got = m(ids[:, 4:], cache, 4)
    assert seen[:-1] == ([(512, "add2")] if B <= 16 else [(512, "bias"), (2048, "add2")]) * 2
    monkeypatch.undo()
    one = torch.cat([m(ids[b:b + 1], None)[:, -1:] for b in range(B)])  # the whole sequence at once: roundings at other places of the same layers
    assert (got.float() - one.float()).abs().max() <= 2.0 ** -5 * one.float().abs().max()


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("P,steps", [(1, 2), (9, 8), (30, 35)])
def test_replies_say_where_they_are(cuda, monkeypatch, P, steps, int8):
    """The steps of a reply read their position on the device; the launches are chosen by the middle of the positions they will be at."""
    from ohara_amd import ops

    m = _phi(cuda)
    prompt = torch.randint(0, 96, (2, P), generator=torch.Generator().manual_seed(P)).to(cuda)
    seen, call = [], ops.phi_attn_linear

    def spy(*args, **kw):
        seen.append((args[9], args[13] is not None))
        return call(*args, **kw)

    monkeypatch.setattr(ops, "phi_attn_linear", spy)
    plain = m.generate_greedy(prompt, steps, use_graph=False, int8=int8)
    if P > 1:  # (a prompt of one token goes through the same call)
        assert set(seen) == {(P + (steps - 1) // 2, True)}
    assert torch.equal(m.generate_greedy(prompt, steps, int8=int8), plain)
