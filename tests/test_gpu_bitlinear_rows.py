"""BitLinears over many rows: quantised once and multiplied in tiles, against the same rows in calls of at most 64 (the kernels that
quantise in their own LDS) and against whole-number products on the CPU.  Everything is compared bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _inputs(cuda, rows, n, k, seed):
    g = torch.Generator(device=cuda).manual_seed(seed)
    x = (torch.randn(rows, k, generator=g, device=cuda) * 2).to(BF)
    t = torch.randint(-1, 2, (n, k), generator=g, device=cuda, dtype=torch.int8)
    nw = (1 + 0.2 * torch.randn(k, generator=g, device=cuda)).to(BF)
    pre = (1 + 0.2 * torch.randn(k, generator=g, device=cuda)).to(BF)
    res = torch.randn(rows, n, generator=g, device=cuda).to(BF)
    return x, t, nw, pre, res


# one tile and parts of one, K below / at / past a step of 256 and off 16, columns off a strip and off four, both tile sizes
@pytest.mark.parametrize("rows,n,k", [(66, 16, 8), (130, 70, 264), (100, 64, 256), (300, 2048, 5632), (193, 130, 1000),
                                      (257, 96, 520), (2050, 5632, 2048), (1000, 6150, 136)])
def test_rows_match_short_calls_and_whole_number_products(cuda, rows, n, k):
    from ohara_amd import ops

    x, t, nw, pre, res = _inputs(cuda, rows, n, k, rows + n + k)
    w = ops.pack_ternary(t, 0.013)
    got, acc = ops.bitlinear(x, nw, w, 1e-5, residual=res, want_acc=True, pre_norm_w=pre)
    step = 60  # no call of one row: that one is quantised by a whole workgroup, with sums in another order
    parts = [ops.bitlinear(x[r:r + step], nw, w, 1e-5, residual=res[r:r + step], want_acc=True, pre_norm_w=pre)
             for r in range(0, rows, step)]
    assert torch.equal(acc, torch.cat([p[1] for p in parts]))
    assert torch.equal(got, torch.cat([p[0] for p in parts]))
    q, s, sq = ops.act_quant_sets(x, [nw], 1e-5, pre)
    at = torch.arange(0, rows, max(1, rows // 64), device=cuda)
    codes = q[0, at, :k].cpu().to(torch.int32)
    assert torch.equal(codes.sum(1).int(), sq[0, at].cpu())
    assert torch.equal(acc[at].cpu(), codes @ t.cpu().to(torch.int32).t())


def test_sets_share_rows_and_keep_their_own_codes(cuda):
    from ohara_amd import ops

    x, t, nw, pre, _ = _inputs(cuda, 211, 352, 264, 3)
    x2, t2, nw2, _, _ = _inputs(cuda, 211, 352, 264, 4)
    a, b = (ops.pack_ternary(t, 0.02), ops.pack_ternary(t2, 0.005))
    one, two = ops.bitlinear_many(x, pre, [(nw, a), (nw2, b)], 1e-5)
    assert torch.equal(one, ops.bitlinear(x, nw, a, 1e-5, pre_norm_w=pre))
    assert torch.equal(two, ops.bitlinear(x, nw2, b, 1e-5, pre_norm_w=pre))


def test_weights_of_another_width_are_refused(cuda):
    """On the host: the launch would read past the weights' end."""
    from ohara_amd import ops

    x, t, nw, pre, _ = _inputs(cuda, 70, 64, 264, 5)
    a, narrow, short = (ops.pack_ternary(w.contiguous(), 0.02) for w in (t, t[:32], t[:, :256]))
    for w in (narrow, short):
        with pytest.raises(ValueError):
            ops.bitlinear_many(x, pre, [(nw, a), (nw, w)], 1e-5)
        kc, vc, cs = torch.zeros(1, 80, 2, 32, dtype=BF, device=cuda), torch.zeros(1, 80, 2, 32, dtype=BF, device=cuda), torch.zeros(80, 16, dtype=BF, device=cuda)
        with pytest.raises(ValueError):
            ops.bitlinear_qkv_rope_append(x, pre, [(nw, a), (nw, w), (nw, a)], 1e-5, 2, 2, 32, cs, cs, 0, kc, vc, seq_len=70)
        assert (kc == 0).all()


@pytest.mark.parametrize("batch,seq,h,h_kv,dh", [(1, 70, 2, 2, 64), (3, 50, 4, 2, 128), (2, 129, 2, 1, 8)])
def test_query_key_value_with_rotary_and_append(cuda, batch, seq, h, h_kv, dh):
    from ohara_amd import ops
    from ohara_amd.llama import rope_tables

    k, t_max, pos = 264, 512, 37
    x, _, _, pre, _ = _inputs(cuda, batch * seq, 8, k, 9)
    projs = []
    for i, heads in enumerate((h, h_kv, h_kv)):
        _, t, nw, _, _ = _inputs(cuda, 1, heads * dh, k, 20 + i)
        projs.append((nw, ops.pack_ternary(t, 0.01 * (i + 1))))
    cos, sin = (c.to(cuda, BF) for c in rope_tables(dh, t_max, 10000.0))
    kc, vc, kr, vr = (torch.zeros(batch, t_max, h_kv, dh, device=cuda, dtype=BF) for _ in range(4))
    got = ops.bitlinear_qkv_rope_append(x, pre, projs, 1e-5, h, h_kv, dh, cos, sin, pos, kc, vc, seq_len=seq)
    want, kk, vv = (ops.bitlinear(x, nw, w, 1e-5, pre_norm_w=pre) for nw, w in projs)
    ops.rope_append(want, kk, vv, batch, seq, h, h_kv, dh, cos, sin, pos, kr, vr)
    assert torch.equal(got, want) and torch.equal(kc, kr) and torch.equal(vc, vr)


@pytest.mark.parametrize("width,batch,seq", [(6, 1, 70), (10, 3, 40), (12, 2, 65)])
def test_prompt_of_a_model_whose_heads_are_not_in_fours(cuda, width, batch, seq):
    """More than 64 rows take any even head width: the tiled launch those in fours, three BitLinears and the rotary launch the others."""
    from ohara_amd.bitnet import BitLlama
    from ohara_amd.llama import Config
    from oracle import bitlinear_ref as BL
    from oracle import llama_ref as R

    kw = dict(vocab_size=96, hidden_size=8 * width, intermediate_size=136, num_attention_heads=8, num_key_value_heads=4,
              num_hidden_layers=2, max_sequence_length=80, rope_theta=10000.0)
    rcfg = R.RefConfig(**kw)
    w = BL.init_ternary_weights(rcfg, seed=3, dtype=BF, gamma=0.05)
    ref, model = R.RefLlama(rcfg, w), BitLlama(Config(**kw), w, device=cuda)
    ids = torch.randint(0, 96, (batch, seq), generator=torch.Generator().manual_seed(seq))
    rc, cache = ref.build_kv_cache(batch), model.build_kv_cache(batch)
    want, got = ref(ids, rc, 0).float(), model(ids.to(cuda), cache, 0).float().cpu()
    # an int8 code that rounds the other way moves its whole row: the bounds of the small ternary models
    scale, d = want.abs().max().item(), (got - want).abs()
    assert d.max().item() <= 8e-2 * scale and d.mean().item() <= 1e-2 * scale
    assert (cache[0].key[:, seq:] == 0).all() and (cache[0].key[:, :seq].float().abs().amax((2, 3)) > 0).all()


@pytest.mark.parametrize("rows", [12, 13, 17, 64, 65])
def test_rows_around_the_change_of_kernel(cuda, rows):
    """A few rows are quantised by every workgroup, more once and multiplied in tiles: the same codes and whole sums, so the same bits
    as the rows give a few at a time."""
    from ohara_amd import ops

    g = torch.Generator().manual_seed(rows)
    H, D, K, N = 2, 64, 264, 200
    x = torch.randn(rows, K, generator=g).to(torch.bfloat16).to(cuda)
    nw = (1 + 0.1 * torch.randn(4, K, generator=g)).to(torch.bfloat16).to(cuda)
    ws = [ops.pack_ternary(torch.randint(-1, 2, (n, K), generator=g, dtype=torch.int8).to(cuda), 0.02) for n in (H * D, H * D, H * D, N)]
    res = torch.randn(rows, N, generator=g).to(torch.bfloat16).to(cuda)
    got = ops.bitlinear(x, nw[3], ws[3], residual=res)
    want = torch.cat([ops.bitlinear(x[i:i + 6], nw[3], ws[3], residual=res[i:i + 6]) for i in range(0, rows, 6)])
    assert torch.equal(got, want)
    angle = torch.rand(128, D // 2, generator=g)
    cos, sin = angle.cos().to(torch.bfloat16).to(cuda), angle.sin().to(torch.bfloat16).to(cuda)
    kc, vc, kp, vp = (torch.zeros(1, 80, H, D, dtype=torch.bfloat16, device=cuda) for _ in range(4))
    projs = [(nw[i], ws[i]) for i in range(3)]
    q = ops.bitlinear_qkv_rope_append(x, nw[3], projs, 1e-5, H, H, D, cos, sin, 3, kc, vc, seq_len=rows)
    parts = [ops.bitlinear_qkv_rope_append(x[i:i + 6], nw[3], projs, 1e-5, H, H, D, cos, sin, 3 + i, kp, vp, seq_len=min(6, rows - i))
             for i in range(0, rows, 6)]
    assert torch.equal(q, torch.cat(parts)) and torch.equal(kc, kp) and torch.equal(vc, vp)
