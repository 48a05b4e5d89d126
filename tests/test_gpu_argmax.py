"""Greedy selection: the first index of the largest value among the valid ids, whatever the values; a NaN is never chosen while there is a
number."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
INF, NAN = float("inf"), float("nan")


def _first_largest(row):
    best, at = None, 0
    for i, v in enumerate(row):
        if v == v and (best is None or v > best):
            best, at = v, i
    return at


def _rows(V):
    """Rows whose answer is not obvious, as bf16 patterns."""
    g = torch.Generator().manual_seed(V)
    wide = torch.randn(V, generator=g).to(BF)
    rows = [wide, torch.zeros(V).to(BF), -wide.abs() - 1, torch.full((V,), -INF).to(BF), torch.full((V,), NAN).to(BF), -torch.full((V,), NAN).to(BF)]

    def spots(base, *at):
        r = base.clone()
        for i, v in at:
            r[i % V] = v
        rows.append(r)

    spots(-wide.abs() - 1, (V - 1, -0.0))                            # the largest is a negative zero, in the tail
    spots(-wide.abs() - 1, (V - 1, 0.0), (V // 2, -0.0), (V // 3 + 1, -0.0))  # zeros of both signs: the same value
    spots(-wide.abs() - 1, (V // 2, 0.0), (V - 2, -0.0))
    spots(wide, (V // 2, INF), (V // 5, INF), (V - 1, INF))
    spots(wide, (0, NAN), (V // 2, -NAN), (V - 1, NAN))
    spots(wide, (V - 1, -NAN), (V // 3, 9.0), (V // 3 + 1, 9.0))
    spots(torch.full((V,), NAN).to(BF), (V - 1, -INF), (V // 2, -INF))
    spots(-torch.full((V,), NAN).to(BF), (V // 2, -INF))
    spots(torch.full((V,), -INF).to(BF), (V - 1, -3.0e38))
    signalling = wide.view(torch.int16).clone()
    signalling[V // 4] = 0x7F81
    rows.append(signalling.view(BF))
    return torch.stack(rows)


@pytest.mark.parametrize("V,pad", [(1, 7), (7, 1), (8, 0), (9, 7), (64, 0), (1000, 0), (8191, 1), (8193, 7), (32000, 0), (65536, 0), (65543, 1), (70001, 7), (131080, 0), (1000, 1)])
def test_first_index_of_the_largest(cuda, V, pad):
    """pad: rows on 16 bytes, or not."""
    from ohara_amd import ops

    rows = _rows(V)
    B = rows.shape[0]
    buf = torch.full((B, V + pad), 1e30).to(BF)
    buf[:, :V] = rows
    for valid in {V, max(1, V - 3), max(1, V // 2)}:
        got = ops.argmax(buf.to(cuda), valid_vocab=valid).tolist()
        assert got == [_first_largest(r[:valid].float().tolist()) for r in rows]
