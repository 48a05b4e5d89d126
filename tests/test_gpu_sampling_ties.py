"""The draw from a table of bf16 patterns where many ids share one: the j-th of them in id order, wherever they lie, for row lengths of every
instance and tails that fill no eighth, among numbers that are none."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("V,valid", [(8192, 0), (8192, 8187), (32000, 31999), (32768, 0), (50008, 50001), (65536, 0), (65536, 65529), (65536, 9)])
@pytest.mark.parametrize("nans", [0, 50])
@pytest.mark.parametrize("temperature", [1.0, 0.7])
def test_which_of_the_ties_is_drawn(cuda, V, valid, nans, temperature):
    from ohara_amd import ops

    g = torch.Generator().manual_seed(V + valid + nans)
    n = valid or V
    sizes = [1, 2, min(n - 1, 7), n // 3, n - 1]
    x, none = torch.full((len(sizes), V), -30.0), torch.zeros(len(sizes), V, dtype=torch.bool)
    u, want = torch.empty(len(sizes)), []
    for row, size in enumerate(sizes):
        at = torch.randperm(n, generator=g)
        if nans:
            none[row, at[size:size + min(nans, n - size - 1)]] = True
        ties = at[:size].sort().values
        x[row, ties] = 5.0  # e^35 times the others': they never reach a thousandth of a tie's share
        j = int(torch.randint(0, size, (1,), generator=g))
        u[row] = (j + 0.5) / size
        want.append(int(ties[j]))
    x[:, n:] = 40.0  # masked
    # the nucleus holds every tie (top_p close to 1): its mass is theirs
    x = x.to(BF)
    x.view(torch.int16)[none] = -1  # the pattern that sorts below every number
    got = ops.sample_topk_topp(x.to(cuda), temperature, 0, 0.9999999, u.to(cuda), valid_vocab=valid or None)
    assert got.tolist() == want


@pytest.mark.parametrize("V", [8192, 40000, 65536])
def test_rows_of_one_value(cuda, V):
    from ohara_amd import ops

    x = torch.full((3, V), 1.5, dtype=BF, device=cuda)
    x.view(torch.int16)[1, 5::7] = -1
    x.view(torch.int16)[2] = -1
    u = torch.tensor([0.25, 0.5, 0.5], device=cuda)
    got = ops.sample_topk_topp(x, 1.0, 0, 0.5, u).tolist()
    # half of the ids are kept, lowest first; an fp32 product decides, so a neighbour or two may be drawn
    assert abs(got[0] - V // 8) <= 2
    live = [i for i in range(V) if i % 7 != 5]
    assert min(abs(got[1] - i) for i in live[len(live) // 4 - 2:len(live) // 4 + 3]) == 0
    assert got[2] == 0
