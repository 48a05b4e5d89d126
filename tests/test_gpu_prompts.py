"""Prompts of different lengths in one call against the same prompts one by one: their rows of the caches, the rows behind them and of other
slots, and the logits of their last tokens."""

import dataclasses

import pytest
import torch

from oracle import llama_ref as R

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _model(cuda, heads, kv_heads, width, layers=2, **kw):
    from ohara_amd.llama import Config, Llama

    kw = dict(vocab_size=640, hidden_size=width, intermediate_size=2 * width, num_attention_heads=heads, num_key_value_heads=kv_heads,
              num_hidden_layers=layers, max_sequence_length=512, **kw)
    fields = {f.name for f in dataclasses.fields(R.RefConfig)}
    kw = {k: v for k, v in kw.items() if k in fields}
    return Llama(Config(**kw), R.init_weights(R.RefConfig(**kw), seed=5, dtype=BF, std=0.06, norm_jitter=0.1), device=cuda)


def _ids(lens, seed=1):
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(0, 640, (n,), generator=g) for n in lens]


# (heads, key heads, width): heads of 128 and 64, and pairs of (prompt, head) that do and do not divide by eight
@pytest.mark.parametrize("heads,kv_heads,width", [(3, 3, 384), (8, 2, 512), (4, 2, 512)])
@pytest.mark.parametrize("lens", [[65, 64], [1, 70], [300, 1, 16, 129, 511, 63, 64, 66], [512, 500, 480, 470, 490], [33] * 9])
def test_prompts_side_by_side(cuda, heads, kv_heads, width, lens):
    m = _model(cuda, heads, kv_heads, width)
    n, prompts = len(lens), _ids(lens)
    slots = [(3 * i + 1) % (n + 2) for i in range(n)] if (n + 2) % 3 else list(range(n, 0, -1))
    cache, alone = m.build_kv_cache(n + 2), m.build_kv_cache(n + 2)
    for c in cache:
        c.key.fill_(7.0)
        c.value.fill_(7.0)
    got = m.prompts(prompts, cache, slots)
    for i, (p, b) in enumerate(zip(prompts, slots)):
        views = [c._row_view(b) for c in alone]
        for v in views:
            v.length = 0
        want = m(p.view(1, -1).to(cuda), views, 0, last_only=True)[0, 0]
        # up to 64 rows alone take kernels that add K in another order; more, the same
        tol = 0.0 if lens[i] > 64 else 2.0 ** -6
        assert (got[i].float() - want.float()).abs().max() <= tol * want.float().abs().max()
        for c, a in zip(cache, alone):
            for x, y in ((c.key[b], a.key[b]), (c.value[b], a.value[b])):
                assert (x[:lens[i]].float() - y[:lens[i]].float()).abs().max() <= tol * y.float().abs().max()
                assert (x[lens[i]:] == 7.0).all()
    for c in cache:
        for b in set(range(n + 2)) - set(slots):
            assert (c.key[b] == 7.0).all() and (c.value[b] == 7.0).all()


# a product of the layer is in parts of its depth alone (768 columns and 768 and 1536 deep; 1024 and 1024 and 2048; 512 and 2048) and whole
# side by side, where there is no room for them
@pytest.mark.parametrize("heads,width,inner", [(6, 768, 1536), (8, 1024, 2048), (4, 512, 2048)])
def test_prompts_side_by_side_of_wider_models(cuda, heads, width, inner):
    from ohara_amd._lib import lib

    kw = dict(vocab_size=640, hidden_size=width, intermediate_size=inner, num_attention_heads=heads, num_key_value_heads=heads, num_hidden_layers=2,
              max_sequence_length=512)
    from ohara_amd.llama import Config, Llama

    m = Llama(Config(**kw), R.init_weights(R.RefConfig(**kw), seed=5, dtype=BF, std=0.06, norm_jitter=0.1), device=cuda)
    lens = [70, 100, 300, 129]
    assert any(lib().ohara_gemm_residual_norm_bytes(n, width, k) for n in lens for k in (width, inner))
    cache, alone, prompts = m.build_kv_cache(4), m.build_kv_cache(4), _ids(lens)
    got = m.prompts(prompts, cache, [2, 0, 3, 1])
    for i, (p, b) in enumerate(zip(prompts, [2, 0, 3, 1])):
        want = m(p.view(1, -1).to(cuda), [c._row_view(b) for c in alone], 0, last_only=True)[0, 0]
        # as for up to 64 rows above: fp32 sums in another order, rounded to 8 bits at the same places of two layers
        tol = 2.0 ** -6
        assert (got[i].float() - want.float()).abs().max() <= tol * want.float().abs().max()
        for c, a in zip(cache, alone):
            for x, y in ((c.key[b], a.key[b]), (c.value[b], a.value[b])):
                assert (x[:lens[i]].float() - y[:lens[i]].float()).abs().max() <= tol * y.float().abs().max()


def test_what_is_refused(cuda):
    m = _model(cuda, 4, 2, 512)
    cache = m.build_kv_cache(3)
    for lens, slots in (([30, 30], [0, 1]), ([100, 0], [0, 1]), ([513, 1], [0, 1]), ([100, 1], [1, 1]), ([100, 1], [0, 3]), ([100], [0, 1])):
        with pytest.raises(ValueError):
            m.prompts(_ids(lens), cache, slots)
    # (all refused on the host: the launches behind would follow pointers and strides that are not there)
    short = _model(cuda, 4, 2, 512).build_kv_cache(3)
    short[1].key, short[1].value = short[1].key[:, :256].contiguous(), short[1].value[:, :256].contiguous()
    for caches in (cache[:1], cache + cache[:1], [], short, m.build_kv_cache(3, int8=True)):
        with pytest.raises(ValueError):
            m.prompts(_ids([70, 9]), caches, [0, 1])
    with pytest.raises(ValueError):
        m.prompts(_ids([70, 9]), cache, [0, 1, 1])
    assert all((c.key == 0).all() for c in cache)
    assert not m.takes_prompts(m.build_kv_cache(2, int8=True))


@pytest.mark.parametrize("bad", [-1, 640])
def test_ids_outside_the_vocabulary(cuda, bad):
    m = _model(cuda, 4, 2, 512)
    cache, prompts = m.build_kv_cache(2), _ids([60, 9])
    prompts[1][4] = bad
    with pytest.raises(IndexError):
        m.prompts(prompts, cache, [0, 1])
    assert all((c.key == 0).all() for c in cache)
    from ohara_amd.batching import ContinuousBatcher

    # a batcher takes it as 0, one prompt or several
    together, apart, zero = (ContinuousBatcher(m, 2) for _ in range(3))
    first = together.add_many(prompts)
    assert first == [apart.add(p) for p in prompts]
    prompts[1][4] = 0
    assert first == zero.add_many(prompts)


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("most", [100, 16384])
def test_batcher_joins_many_at_once(cuda, monkeypatch, int8, most):
    """All together, in groups and one by one: the same first tokens and the same steps after them."""
    from ohara_amd.batching import ContinuousBatcher

    monkeypatch.setattr(ContinuousBatcher, "GROUP_ROWS", most)
    m = _model(cuda, 4, 2, 512)
    prompts = _ids([70, 3, 90, 200, 5, 65], seed=9)
    together, apart = (ContinuousBatcher(m, 8, int8=int8) for _ in range(2))
    first = together.add_many(prompts)
    assert first == [apart.add(p) for p in prompts]
    assert together.lengths == apart.lengths and together.seq_pos.tolist() == apart.seq_pos.tolist()
    assert [c.lengths for c in together.cache] == [c.lengths for c in apart.cache]
    assert together.steps(5) == apart.steps(5)
    assert together.add_many([]) == []


def test_feed_of_nothing(cuda):
    from ohara_amd.batching import ContinuousBatcher

    b = ContinuousBatcher(_model(cuda, 4, 2, 512), 3)
    assert b.feed([]) == []
    slot, tok = b.add(_ids([70])[0])
    assert b.feed([]) == [] and b.lengths[slot] == 70
    assert [s for s, _ in b.feed([(slot, [tok])])] == [slot]
