"""Tier assignment: scores -> ``tiers[S]`` (fade/policy.py:232-274).

Host-side policy logic (an argsort of at most a few thousand scores per
layer), kept in torch exactly as the reference computes it; the tiers it
returns drive ``TieredKVCache.apply_tier_assignment``.
"""

from __future__ import annotations

import numpy as np
import torch
from torch import Tensor

from ._lib import plain
from .cache import TIER_EVICT, TIER_FP16, TIER_INT2, TIER_INT4


def _assign_one_layer(
    S: int,
    scores: Tensor,
    n_sink: int,
    recent_window: int,
    int4_budget: int | None,
    int2_budget: int,
) -> Tensor:
    """Sinks and the recent window stay FP16; the middle is ranked by score.

    ``int4_budget=None`` keeps every middle token in INT4 (no eviction).
    Otherwise the top ``int4_budget`` scores go to INT4, the next
    ``int2_budget`` to INT2 and the rest are evicted.
    """
    sink_end = min(n_sink, S)
    # the middle is one range: everything between the sinks and the recent window
    lo = sink_end if sink_end >= 0 else max(0, S + sink_end)
    hi = min(S, max(sink_end, S - recent_window))
    tiers = torch.full((S,), TIER_FP16, dtype=torch.long, device=scores.device)
    n = hi - lo
    if n <= 0:
        return tiers
    middle = tiers[lo:hi]
    if int4_budget is None or int4_budget >= n:
        middle.fill_(TIER_INT4)
        return tiers
    middle.fill_(TIER_EVICT)
    k2 = max(0, min(int2_budget, n - int4_budget))
    masks = _top_masks(scores, lo, hi, int4_budget, k2)
    if masks is not None:
        out = middle.numpy()
        out[masks[0]] = TIER_INT4
        if k2 > 0:
            out[masks[1]] = TIER_INT2
        return tiers
    order = scores[torch.arange(lo, hi, device=scores.device)].argsort(descending=True)
    middle[order[:int4_budget]] = TIER_INT4
    if k2 > 0:
        middle[order[int4_budget : int4_budget + k2]] = TIER_INT2
    return tiers


def _top_masks(scores: Tensor, lo: int, hi: int, k1: int, k2: int):
    """Masks over ``scores[lo:hi]`` of its ``k1`` largest values and of the ``k2`` after
    them, by selection instead of a sort (the rule over 4096 host scores: 260 -> 64 us); None where
    a sort has to decide: device scores, equal values across a boundary, NaN, tensors that are
    no plain memory or are being traced."""
    if scores.device.type != "cpu" or scores.dim() != 1 or int(scores.shape[0]) < hi or k1 < 0:
        return None
    scores = scores.detach()
    if scores.dtype not in (torch.float32, torch.float64) or not plain(scores):
        return None
    s = scores[lo:hi].numpy()
    cuts = [c for c in (s.size - k1, s.size - k1 - k2) if c < s.size]
    part = np.partition(s, cuts) if cuts else s
    top = s >= part[s.size - k1] if k1 > 0 else np.zeros(s.size, dtype=bool)
    both = s >= part[s.size - k1 - k2] if k2 > 0 else top
    if np.count_nonzero(top) != k1 or np.count_nonzero(both) != k1 + k2:
        return None
    return top, both & ~top


def reassign_tiers_by_position(cache, num_layers: int) -> None:
    """Position (FIFO) policy: newer middle tokens score higher (fade/policy.py:126-159)."""
    for li in range(num_layers):
        if not cache.is_managed(li):
            continue
        S = int(cache.get_seq_length(li))
        if S == 0:
            continue
        scores = torch.arange(S, dtype=torch.float32)
        tiers = _assign_one_layer(S, scores, cache.n_sink, cache.recent_window, cache.int4_budget, cache.int2_budget)
        cache.apply_tier_assignment(li, tiers)


def reassign_tiers_with_scores(cache, layer_scores: dict[int, Tensor]) -> None:
    """Apply the rule to externally computed per-layer scores (e.g. H2O attention mass)."""
    for li, scores in layer_scores.items():
        S = cache.get_seq_length(li)
        tiers = _assign_one_layer(S, scores, cache.n_sink, cache.recent_window, cache.int4_budget, cache.int2_budget)
        cache.apply_tier_assignment(li, tiers, scores=scores)


__all__ = ["_assign_one_layer", "reassign_tiers_by_position", "reassign_tiers_with_scores"]
