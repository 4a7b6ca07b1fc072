"""The packed decode's automatic split count, and the split merge of the general kernel,
around the sizes where the split count changes: against the same call in one split."""

from __future__ import annotations

import pytest
import torch

from fade_amd.kernels import MiddleTier, tiered_decode_attention
from fade_amd.quant import quant_asym, quant_k_int4, quant_v_int4

pytestmark = pytest.mark.gpu


def _call(dev, B, Hq, Hkv, D, S, dtype, fmt):
    g = torch.Generator().manual_seed(B * 1000 + S)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)  # noqa: E731
    k, v = rnd(B, Hkv, S, D), rnd(B, Hkv, S, D)
    if fmt == "asym":
        (kq, ks, kz), (vq, vs, vz) = quant_asym(k, 4), quant_asym(v, 2)
        mid = MiddleTier("asym", kq, vq, ks, vs, kz, vz, k_bits=4, v_bits=2, group=32)
    else:
        (kq, ks), (vq, vs) = quant_k_int4(k), quant_v_int4(v)
        mid = MiddleTier("int4", kq, vq, ks, vs)
    q, sink, rec = rnd(B, Hq, 1, D), (rnd(B, Hkv, 4, D), rnd(B, Hkv, 4, D)), (rnd(B, Hkv, 40, D), rnd(B, Hkv, 40, D))
    return lambda **kw: tiered_decode_attention(q, sink, mid, rec, **{"deterministic": True, **kw}).float()


# one tile; a few tiles of one (row, head); about a tile per wave and split; more splits than
# the merge takes at once; two workgroups per CU
@pytest.mark.parametrize("B,Hq,Hkv,S", [(1, 4, 1, 30), (1, 4, 1, 300), (1, 32, 8, 600), (1, 32, 8, 2048), (1, 8, 2, 9000), (16, 32, 8, 1030)])
@pytest.mark.parametrize("dtype,fmt", [(torch.float16, "int4"), (torch.bfloat16, "int4"), (torch.float16, "asym")])
def test_packed_auto_splits(dev, B, Hq, Hkv, S, dtype, fmt):
    run = _call(dev, B, Hq, Hkv, 128, S, dtype, fmt)
    # each probability is rounded to 16 bits against its own split's maximum
    tol = (2e-3, 0) if dtype == torch.float16 else (4e-3, 2.0**-7)
    one = run(n_splits=1)
    assert bool(((run() - one).abs() <= tol[0] + tol[1] * one.abs()).all())


# 1024 / D splits at a time, four rounds of them ahead of the maximum, then one by one
@pytest.mark.parametrize("D,n", [(64, 1), (64, 16), (64, 17), (64, 65), (256, 5), (256, 17), (80, 12), (80, 49), (8, 3)])
def test_general_kernel_split_merge(dev, D, n):
    run = _call(dev, 2, 4, 2, D, 64 * 70, torch.float16, "int4")
    one = run(n_splits=1)
    assert bool(((run(n_splits=n) - one).abs() <= 2e-3).all())


# calls whose slot-filling split count leaves every wave one tile: the split count that is taken
# instead keeps it so, and no claim order or split count enters a probability's rounding
@pytest.mark.parametrize("B,Hq,Hkv,S", [(1, 4, 1, 300), (1, 32, 8, 2048), (4, 32, 8, 1030), (2, 28, 4, 1334)])
@pytest.mark.parametrize("dtype,fmt", [(torch.float16, "int4"), (torch.bfloat16, "int4"), (torch.float16, "asym")])
def test_small_calls_repeat(dev, B, Hq, Hkv, S, dtype, fmt):
    run = _call(dev, B, Hq, Hkv, 128, S, dtype, fmt)
    fixed, most = run(), run(n_splits=10**4)  # in tiles order; one tile per split
    ulp = 2.0**-10 if dtype == torch.float16 else 2.0**-7
    assert bool(((fixed - most).abs() <= ulp * most.abs() + 1e-6).all())  # the fp32 merge's order only
    for _ in range(3):
        assert torch.equal(run(deterministic=False), fixed)
