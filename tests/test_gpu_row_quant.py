"""A workgroup a row, or a wave: the codes of the kernel that gives a row a wave, bit for bit, for every number of pieces a thread holds, one to three
norms at once, and rows that are multiplied out of gate and up on the way."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
DEPTHS = [8, 72, 520, 2048, 2056, 4096, 4104, 5632, 6144]


@pytest.mark.parametrize("k", DEPTHS)
@pytest.mark.parametrize("rows,sets", [(2, 1), (13, 3), (300, 2)])
def test_codes_of_rows(cuda, k, rows, sets):
    from ohara_amd import ops

    g = torch.Generator(device=cuda).manual_seed(k + rows)
    n = lambda *s: (torch.randn(*s, generator=g, device=cuda) * 2).to(BF)  # noqa: E731
    wide = n(rows, k + 8)
    x, norms, pre = wide[:, :k].contiguous(), [n(k) for _ in range(sets)], n(k)
    x[0] = 0
    x[1, k // 2] = float("inf")
    norms[0][k - 1] = float("nan")
    q, s, sq = ops.act_quant_sets(x, norms, 1e-5)
    for i, w in enumerate(norms):
        want = ops.act_quant(x, w)
        assert torch.equal(q[i, :, :k], want[0][:, :k]) and torch.equal(s[i], want[1]) and torch.equal(sq[i], want[2])
    # a block norm ahead: rms over a sum of squares of the rounded row
    x[1, k // 2] = 1.0
    q, s, sq = ops.act_quant_sets(x, norms, 1e-5, pre)
    once = ops.act_quant_sets(x, norms[-1:], 1e-5, pre)
    assert torch.equal(q[-1, :, :k], once[0][0, :, :k]) and torch.equal(s[-1], once[1][0]) and torch.equal(sq[-1], once[2][0])
    normed = ops.rmsnorm(x, pre)
    plain = ops.act_quant(normed, norms[-1])
    off = (q[-1, :, :k].int() - plain[0][:, :k].int()).abs()  # (the norm's own sum is in another order: a code may move by one)
    assert off.max() <= 1 and (off > 0).float().mean() < 0.01


@pytest.mark.parametrize("k", DEPTHS)
@pytest.mark.parametrize("rows", [2, 65])
def test_gate_and_up_on_the_way(cuda, k, rows):
    from ohara_amd import ops
    from ohara_amd._lib import check, lib

    g = torch.Generator(device=cuda).manual_seed(k * rows)
    n = lambda *s: torch.randn(*s, generator=g, device=cuda)  # noqa: E731
    gate, up, w = (n(rows, k) * 40).to(BF), n(rows, k).to(BF), n(k).to(BF)
    want = ops.act_quant_sets(ops.silu_mul(gate, up), [w], 1e-5)
    ldq = (k + 15) // 16 * 16
    q, s, sq = torch.empty(rows, ldq, dtype=torch.int8, device=cuda), torch.empty(rows, device=cuda), torch.empty(rows, dtype=torch.int32, device=cuda)
    st = torch.cuda.current_stream().cuda_stream
    check(lib().ohara_act_quant_swiglu_int8(gate.data_ptr(), up.data_ptr(), k, w.data_ptr(), 1e-5, rows, k, q.data_ptr(), ldq, s.data_ptr(),
                                            sq.data_ptr(), st), "act_quant_swiglu")
    assert torch.equal(q[:, :k], want[0][0, :, :k]) and torch.equal(s, want[1][0]) and torch.equal(sq, want[2][0])
    assert lib().ohara_act_quant_swiglu_int8(gate.data_ptr(), up.data_ptr(), k - 1, w.data_ptr(), 1e-5, rows, k, q.data_ptr(), ldq, s.data_ptr(),
                                             sq.data_ptr(), st) != 0


@pytest.mark.parametrize("k,rows", [(8, 5), (504, 13), (512, 1025), (520, 299), (520, 301), (1024, 300), (1032, 1023), (1032, 1027), (2048, 1024), (2056, 1025),
                                    (3072, 1026), (3080, 1024)])
@pytest.mark.parametrize("sets", [1, 3])
def test_a_wave_a_row(cuda, k, rows, sets):
    """On both sides of the lines between the two, rows that do not fill a workgroup among them: the codes of two rows at a time."""
    from ohara_amd import ops
    from ohara_amd._lib import check, lib

    g = torch.Generator(device=cuda).manual_seed(k + rows)
    n = lambda *s: (torch.randn(*s, generator=g, device=cuda) * 2).to(BF)  # noqa: E731
    x, up, norms, pre = n(rows, k), n(rows, k), [n(k) for _ in range(sets)], n(k)
    x[0] = 0
    some = [slice(0, 2), slice(rows - 3, rows - 1), slice(rows - 2, rows)]
    for block_norm in (None, pre):
        q, s, sq = ops.act_quant_sets(x, norms, 1e-5, block_norm)
        for at in some:
            want = ops.act_quant_sets(x[at], norms, 1e-5, block_norm)
            assert torch.equal(q[:, at, :k], want[0][..., :k]) and torch.equal(s[:, at], want[1]) and torch.equal(sq[:, at], want[2])
        if block_norm is None:
            for i, w in enumerate(norms):
                want = ops.act_quant(x, w)
                assert torch.equal(q[i, :, :k], want[0][:, :k]) and torch.equal(s[i], want[1]) and torch.equal(sq[i], want[2])
    want = ops.act_quant_sets(ops.silu_mul(x, up), norms[:1], 1e-5)
    ldq = (k + 15) // 16 * 16
    q, s, sq = torch.empty(rows, ldq, dtype=torch.int8, device=cuda), torch.empty(rows, device=cuda), torch.empty(rows, dtype=torch.int32, device=cuda)
    check(lib().ohara_act_quant_swiglu_int8(x.data_ptr(), up.data_ptr(), k, norms[0].data_ptr(), 1e-5, rows, k, q.data_ptr(), ldq, s.data_ptr(),
                                            sq.data_ptr(), torch.cuda.current_stream().cuda_stream), "act_quant_swiglu")
    assert torch.equal(q[:, :k], want[0][0, :, :k]) and torch.equal(s, want[1][0]) and torch.equal(sq, want[2][0])
