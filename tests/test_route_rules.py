"""Which kernel a call takes, on both sides of the lines (no GPU)."""

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


@pytest.mark.parametrize("rows,k,packed_rows,ahead", [
    (64, 1024, 65536, 0), (65, 1024, 16, 1), (65, 4096, 16, 1),                    # narrow models; many rows
    (32, 1025, 65536, 0), (33, 1032, 2720, 0), (33, 1032, 2736, 1), (48, 1536, 2736, 1), (49, 1536, 2048, 0), (64, 1536, 2064, 1),
    (32, 1544, 65536, 0), (33, 1544, 1360, 0), (33, 2048, 1376, 1), (48, 2048, 1360, 0), (48, 2048, 1376, 1), (64, 2048, 1024, 0), (64, 2048, 1040, 1),
    (16, 2056, 65536, 0), (17, 2056, 16, 1),
])
def test_norms_ahead_of_a_projection(rows, k, packed_rows, ahead):
    from ohara_amd import ops
    from ohara_amd._lib import lib

    assert lib().ohara_projection_norm_ahead(rows, k, packed_rows) == ahead
    assert not ahead or rows > ops.norm_rows(k)
    assert lib().ohara_projection_norm_ahead(0, k, packed_rows) == lib().ohara_projection_norm_ahead(rows, k, 0) == 0


# heads, their width, columns and depth of the product, sequences, chunks asked for, position -> chunks of the one launch (0: two)
@pytest.mark.parametrize("h,dh,n,k,batch,ns,pos,chunks", [
    *((32, 80, 2560, 10240, 1, 16, pos, 12) for pos in (0, 40, 700, 1500, 1750, 2047)),
    (32, 80, 2560, 10240, 2, 8, 40, 0), (32, 80, 2560, 10240, 17, 1, 0, 0), (32, 80, 2560, 2040, 1, 16, 0, 0), (32, 64, 4096, 8192, 1, 16, 0, 0),
    (32, 64, 2048, 8192, 4, 4, 200, 4), (32, 64, 2048, 8192, 4, 4, 1000, 0), (32, 64, 2048, 8192, 4, 4, 1740, 0),
    (32, 64, 2048, 8192, 16, 1, 100, 1), (32, 64, 2048, 8192, 16, 1, 700, 0), (16, 64, 1024, 4096, 1, 16, 40, 16), (16, 64, 1024, 4096, 1, 16, 100, 0),
    (8, 64, 512, 2048, 1, 16, 0, 16), (8, 64, 512, 2048, 1, 16, 100, 0), (8, 64, 512, 2048, 8, 8, 1500, 0), (24, 64, 1536, 6144, 1, 16, 1000, 16),
])
def test_phi_attention_beside_a_product(h, dh, n, k, batch, ns, pos, chunks):
    from ohara_amd import _lib

    of = _lib.lib().ohara_phi_attn_linear_chunks
    assert of(batch, h, dh, ns, pos, n, k) == chunks
    assert of(0, h, dh, ns, pos, n, k) == of(batch, h, dh, 65, pos, n, k) == of(batch, h, dh, ns, -1, n, k) == _lib.EINVAL


# rows, packed rows, depth, epilogue, width of a rotary head -> rows of the first launch
@pytest.mark.parametrize("rows,packed,k,epilogue,dh,first", [
    (8192, 2304, 768, 3, 128, 7168), (16384, 2304, 768, 3, 64, 14336), (8192, 6144, 768, 2, 0, 0), (5421, 2992, 2560, 0, 0, 5376), (1023, 17920, 2560, 0, 0, 0),
    (3615, 5776, 256, 0, 0, 0), (3615, 5776, 256, 4, 0, 0), (1870, 9008, 512, 4, 0, 0), (6209, 5600, 760, 0, 0, 0),
])
def test_rows_of_a_first_launch(rows, packed, k, epilogue, dh, first):
    from ohara_amd import _lib

    of = _lib.lib().ohara_gemm_first_rows
    assert of(rows, packed, k, epilogue, dh) == first
    assert of(0, packed, k, epilogue, dh) == of(rows, packed, k, 12, dh) == of(rows, packed, k, -1, dh) == of(rows, packed, k, 3, 0) == _lib.EINVAL


# rows of 512 tiles of 128 x 192, and of up to 32 fewer: the same tile for both
@pytest.mark.parametrize("full,fewer,packed,k,tile", [(16384, 16256, 768, 768, 256256), (4096, 3900, 3072, 1024, 256256), (16384, 16256, 768, 3072, 256256)])
def test_a_full_round_is_no_quicker_than_one_that_lacks_tiles(full, fewer, packed, k, tile):
    from ohara_amd import _lib

    assert _lib.lib().ohara_gemm_tile_of(full, packed, k) == _lib.lib().ohara_gemm_tile_of(fewer, packed, k) == tile
