"""Which attention kernel a call of a few tokens takes (no GPU)."""

import pytest


@pytest.mark.parametrize("B,S,H,Hkv,D,pos", [(1, 2, 6, 6, 128, 1000), (1, 8, 6, 6, 128, 3000), (1, 2, 16, 16, 64, 2000)])
def test_a_few_tokens_without_room_for_chunks(B, S, H, Hkv, D, pos):
    """What wins only in chunks does not without room for their partial results; sixteen tokens, or walks enough, do either way."""
    from ohara_amd._lib import lib

    room = lib().ohara_attn_prefill_ws_bytes(B, S, H, Hkv, D, pos)
    assert room > 0 and lib().ohara_attn_prefill_wins(B, S, H, Hkv, D, pos) == 1
    assert [lib().ohara_attn_prefill_wins_with(B, S, H, Hkv, D, pos, n) for n in (room, room // 2, 0)] == [1, 0, 0]
    for b, s in ((B, 16), (40, 15)):
        assert lib().ohara_attn_prefill_wins_with(b, s, H, Hkv, D, pos, 0) == lib().ohara_attn_prefill_wins(b, s, H, Hkv, D, pos) == 1
