"""Slots of a ragged batch taken and left in one launch: one, as many as a launch carries, one more, several launches."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 128, 129, 300])
def test_slots_taken_and_left(cuda, n):
    from ohara_amd import ops

    batch = n + 7
    g = torch.Generator().manual_seed(n)
    slots = torch.randperm(batch, generator=g)[:n].tolist()
    positions = torch.randint(0, 4096, (n,), generator=g).tolist()
    ids = torch.randint(0, 2 ** 40, (n,), generator=g).to(cuda)
    pos, flags, last = (torch.randint(1, 100, (batch,), generator=g).to(t).to(cuda) for t in (torch.int32, torch.uint8, torch.int64))
    want = [t.clone() for t in (pos, flags, last)]
    at = torch.tensor(slots, device=cuda)
    want[0][at], want[1][at] = torch.tensor(positions, dtype=torch.int32, device=cuda), 1
    ops.set_slots(slots, positions, pos, flags, last)  # ids as they are
    assert all(torch.equal(a, b) for a, b in zip((pos, flags, last), want))
    want[2][at] = ids
    ops.set_slots(slots, positions, pos, flags, last, ids)
    assert all(torch.equal(a, b) for a, b in zip((pos, flags, last), want))
    for t in want:
        t[at] = 0
    ops.set_slots(slots, None, pos, flags, last)
    assert all(torch.equal(a, b) for a, b in zip((pos, flags, last), want))
    for bad in ([batch], [-1]):
        with pytest.raises((RuntimeError, ValueError)):
            ops.set_slots(bad, [0], pos, flags, last)
    with pytest.raises(ValueError):
        ops.set_slots(slots, positions + [1], pos, flags, last)
