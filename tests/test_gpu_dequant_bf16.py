"""bf16 INT4 dequantization on hardware conversions against torch's bf16 product, bit for bit."""

from __future__ import annotations

import pytest
import torch

from fade_amd import quant as fq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1, 128), (2, 3, 67, 128), (1, 2, 40, 80), (1, 3, 33, 8), (1, 1, 50, 256)])
@pytest.mark.parametrize("per_token", [True, False])
def test_dequant_int4_bf16(dev, shape, per_token):
    B, H, S, D = shape
    g = torch.Generator().manual_seed(S)
    packed = torch.randint(0, 256, (B, H, S, D // 2), generator=g, dtype=torch.uint8)
    codes = torch.stack([packed >> 4, packed & 15], -1).flatten(-2).to(torch.int8)
    codes = torch.where(codes > 7, codes - 16, codes)
    scale = torch.randn((B, H, S, 1) if per_token else (B, H, 1, D), generator=g).bfloat16()
    flat = scale.view(-1)
    special = [float("inf"), float("nan"), 3.0e38, 1e-40, -0.0, 9.2e-41]
    for i, x in enumerate(special):
        flat[(7 * i) % flat.numel()] = x
    want = codes.bfloat16() * scale
    shifted = torch.zeros(flat.numel() + 3, dtype=torch.bfloat16, device=dev)  # a scale off 16-byte alignment
    shifted[3:] = flat.to(dev)
    for s in (scale.to(dev), shifted[3:].view(scale.shape)):
        out = fq.dequant_int4(packed.to(dev), s, dtype=torch.bfloat16).cpu()
        assert torch.equal(out.isnan(), want.isnan())
        assert torch.equal(out.view(torch.int16)[~want.isnan()], want.view(torch.int16)[~want.isnan()])
