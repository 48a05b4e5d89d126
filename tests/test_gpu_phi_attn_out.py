"""Phi's attention of one token beside a product, its chunks merged by the output projection: against 64 bits, over chunks and fours of chunks that begin, fill
and end, replayed from a graph with other positions, with old sums in the workspace; and where the call is refused."""

import pytest
import torch

from test_gpu_phi_attn_linear import _attention

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

# batch, heads, head width, rotated, chunks, rows and depth of the product
SHAPES = [
    (1, 32, 80, 32, 16, 2560, 10240), (2, 32, 80, 32, 8, 2560, 2560), (1, 40, 64, 32, 16, 2560, 2048), (2, 16, 128, 64, 16, 2044, 2056),
    (1, 18, 120, 48, 16, 1000, 2048), (1, 32, 128, 32, 4, 1024, 4096), (2, 64, 32, 16, 4, 512, 2048),
]


@pytest.mark.parametrize("B,H,D,rot,ns,n,k", SHAPES)
def test_merged_by_the_projection(cuda, B, H, D, rot, ns, n, k):
    from ohara_amd import ops
    from ohara_amd.phi import rope_cos_sin

    T, K = 2048, H * D
    g = torch.Generator(device=cuda).manual_seed(H + D + ns + n)
    r = lambda *s: torch.randn(*s, generator=g, device=cuda).to(BF)  # noqa: E731
    q, keys, values, x, bias, w = r(B, K), r(B, T, H, D), r(B, T, H, D), r(B, k), r(n), ops.pack_linear(r(n, k))
    wo, bias_o, add = r(n, K), r(n), r(B, n)
    packed = ops.pack_linear(wo)
    cos, sin = (t.to(cuda) for t in rope_cos_sin(T, rot))
    ws = ops.phi_attn_workspace(B, H, D, ns, cuda)
    after = -(-B * H * 4 // 256) * 256
    alone = ops.linear_bias(x, w, bias)
    y, out = torch.empty(B, n, dtype=BF, device=cuda), torch.empty(B, n, dtype=BF, device=cuda)
    dev = torch.zeros(1, dtype=torch.int32, device=cuda)

    def call(pos, pos_dev):
        ops.phi_attn_out(q, keys, values, cos, sin, rot, B, H, D, pos, x, w, bias, pos_dev, y, ns, ws, packed, bias_o, add, out)

    def check(pos):
        want, bound = (t.reshape(B, K) for t in _attention(q.view(B, H, D), keys, values, cos, sin, rot, pos))
        woT, size = wo.double().t().contiguous(), wo.double().abs().t().contiguous()
        v = want @ woT + bias_o.double()
        # the rows' own bound through the weights, an fp32 sum of K products and the bias, and a rounding to bf16 of each of three sums
        err = bound @ size + ((want.abs() + bound) @ size + bias_o.double().abs()) * (K + 16) * 2.0 ** -24
        for part in (0, alone.double(), add.double()):
            v = v + part
            err = err + (v.abs() + err) * 2.0 ** -8
        assert torch.equal(y, alone)
        assert ((out.double() - v).abs() <= err).all()
        out.fill_(7.0)
        y.fill_(7.0)

    per = [64, 4 * 64, ns * 64]
    places = sorted({p for e in per for p in (e - 1, e, e + 1)} | {0, 15, 64, 100, 500, 900})
    reached = [p for p in places if ops.phi_attn_out_chunks(B, H, D, rot, ns, p, n, k)]
    assert len(reached) >= 5
    for pos in reached:
        ws[after:] = 255  # (not numbers)
        call(pos, None)
        check(pos)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(reached[-1], dev)
    for pos in sorted({*places, 1500, T - 1}):
        ws[after:] = 255
        dev.fill_(pos)
        graph.replay()
        check(pos)
    keys[:, 70, 0, 0] = float("nan")  # the row of that head, and so every column
    dev.fill_(100)
    graph.replay()
    assert out.isnan().all()


def test_refused(cuda):
    from ohara_amd import _lib, ops

    of = ops.phi_attn_out_chunks
    assert of(1, 32, 80, 32, 16, 700, 2560, 10240) == 12 and of(2, 32, 80, 32, 8, 700, 2560, 10240) == 4
    for no in ((3, 32, 80, 32, 8, 700, 2560, 10240), (1, 32, 80, 32, 16, 40, 2560, 10240), (2, 32, 80, 32, 8, 2000, 2560, 10240), (1, 24, 80, 32, 16, 700, 1920, 7680),
               (1, 32, 80, 40, 16, 700, 2560, 10240), (1, 128, 16, 16, 16, 700, 2048, 8192), (1, 32, 80, 32, 3, 700, 2560, 10240), (1, 32, 128, 32, 16, 700, 4096, 8192)):
        assert of(*no) == 0
    assert of(0, 32, 80, 32, 16, 700, 2560, 10240) == of(1, 32, 80, 33, 16, 700, 2560, 10240) == of(1, 32, 80, 32, 16, -1, 2560, 10240) == _lib.EINVAL
    new = lambda *s: torch.zeros(*s, dtype=BF, device=cuda)  # noqa: E731
    q, kv, x, y, bias = new(1, 2560), new(1, 1024, 32, 80), new(1, 2560), new(1, 2560), new(2560)
    w, angles, ws = ops.pack_linear(new(2560, 2560)), torch.zeros(1024, 16, device=cuda), ops.phi_attn_workspace(1, 32, 80, 16, cuda)

    def status(pos=700, ns=16, ws=ws.data_ptr(), ldx=2560, n=2560, out=y.data_ptr(), cos=angles.data_ptr()):
        return _lib.lib().ohara_phi_attn_out_bf16(q.data_ptr(), 2560, kv.data_ptr(), kv.data_ptr(), cos, cos, 32, 1, 32, 80, 1024, pos, None, ns, ws, x.data_ptr(), ldx,
                                                  w.data.data_ptr(), n, 2560, bias.data_ptr(), y.data_ptr(), 2560, w.data.data_ptr(), bias.data_ptr(), y.data_ptr(),
                                                  2560, out, 2560, torch.cuda.current_stream().cuda_stream)

    assert all(s == _lib.EINVAL for s in (status(pos=1024), status(ws=None), status(ws=ws.data_ptr() + 8), status(ldx=2552), status(n=2558), status(out=None)))
    assert status(pos=0) == status(ns=1) == status(cos=angles.data_ptr() + 4) == _lib.ESIZE
    with pytest.raises(ValueError, match="out must"):
        ops.phi_attn_out(q, kv, kv, angles, angles, 32, 1, 32, 80, 700, x, w, bias, None, y, 16, ws, w, bias, y, new(1, 64))
