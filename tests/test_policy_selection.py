"""Tier assignment by selection against the reference's sort (fade/policy.py:232-274)."""

from __future__ import annotations

import pytest
import torch

from fade_amd.policy import TIER_EVICT, TIER_FP16, TIER_INT2, TIER_INT4, _assign_one_layer


def _by_sort(S, scores, n_sink, recent, b4, b2):
    tiers = torch.full((S,), TIER_EVICT, dtype=torch.long)
    sink_end = min(n_sink, S)
    tiers[:sink_end] = TIER_FP16
    tiers[max(sink_end, S - recent) :] = TIER_FP16
    middle = (tiers == TIER_EVICT).nonzero().squeeze(-1)
    if middle.numel() == 0:
        return tiers
    if b4 is None or b4 >= middle.numel():
        tiers[middle] = TIER_INT4
        return tiers
    order = scores[middle].argsort(descending=True)
    tiers[middle[order[:b4]]] = TIER_INT4
    if b2 > 0:
        k2 = min(b2, order.shape[0] - b4)
        if k2 > 0:
            tiers[middle[order[b4 : b4 + k2]]] = TIER_INT2
    return tiers


@pytest.mark.parametrize("S", [0, 1, 5, 70, 4096])
@pytest.mark.parametrize("n_sink,recent", [(0, 0), (4, 64), (4, 0), (0, 3), (100, 100), (2, -1)])
@pytest.mark.parametrize("b4,b2", [(None, 0), (0, 0), (0, 2), (1, 0), (3, 1), (400, 0), (400, 300), (10, 10**6), (10**6, 5)])
def test_assignment_equals_the_sort(S, n_sink, recent, b4, b2):
    g = torch.Generator().manual_seed(S)
    kinds = {
        "float": torch.rand(S, generator=g),
        "double": torch.rand(S, generator=g, dtype=torch.float64),
        "longer": torch.rand(S + 9, generator=g),
        "ties": torch.randint(0, 3, (S,), generator=g).float(),
        "ints": torch.randint(0, 1000, (S,), generator=g),
        "half": torch.rand(S, generator=g).half(),
        "infinite": torch.where(torch.rand(S, generator=g) < 0.3, float("inf"), -float("inf")),
        "nan": torch.where(torch.rand(S, generator=g) < 0.1, float("nan"), torch.rand(S, generator=g)),
        "strided": torch.rand(2 * S, generator=g)[::2],
    }
    for name, s in kinds.items():
        assert torch.equal(_assign_one_layer(S, s, n_sink, recent, b4, b2), _by_sort(S, s, n_sink, recent, b4, b2)), name


def test_scores_shorter_than_the_cache():
    with pytest.raises(IndexError):
        _assign_one_layer(100, torch.rand(50), 4, 4, 10, 0)


def test_scores_that_numpy_does_not_take():
    """Scores with a pending negation, and scores under a recorder: the sort decides, as for other tensors."""
    z = torch.complex(torch.rand(50), torch.rand(50))
    s = z.conj().imag
    assert s.is_neg()
    assert torch.equal(_assign_one_layer(50, s, 4, 4, 10, 5), _by_sort(50, s, 4, 4, 10, 5))
    s = torch.rand(50, requires_grad=True)
    assert torch.equal(_assign_one_layer(50, s, 4, 4, 10, 5), _by_sort(50, s.detach(), 4, 4, 10, 5))
