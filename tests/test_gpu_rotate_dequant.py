"""Fused dequantize + rotate back (``fade_rotate_dequant``, fade/rotated_quant.py:134-145,176-187)
against a 64-bit product of the same dequantized rows."""

from __future__ import annotations

import pytest
import torch

from fade_amd import _lib
from fade_amd import rotated_quant as frq
from fade_amd.quant import dequant_sym

pytestmark = pytest.mark.gpu


def _inputs(shape, bits, axis, dtype, dev, seed=3):
    g = torch.Generator().manual_seed(seed)
    B, H, S, D = shape
    if bits == 3:
        packed = torch.randint(-4, 4, (B, H, S, D), generator=g, dtype=torch.int8)
    else:
        packed = torch.randint(0, 256, (B, H, S, D * bits // 8), generator=g, dtype=torch.uint8)
    sshape = (B, H, 1, D) if axis == _lib.AXIS_CHANNEL else (B, H, S, 1)
    scale = (torch.rand(sshape, generator=g) * 0.5 + 1e-3).to(dtype)
    return packed.to(dev), scale.to(dev)


def _check(packed, scale, R, bits, dtype):
    """|out - exact| <= half an ulp of the output plus the fp32-GEMM term: 128 products summed
    in fp32, each entry of R in its 24 bits."""
    assert frq._dequant_fused_ok(packed, R, bits, dtype)
    out = frq.rotated_dequant_k(packed, scale, R, bits, dtype).double()
    x = dequant_sym(packed, scale, bits, dtype).double()
    ref = x @ R.double()
    half_ulp = 2.0**-11 if dtype == torch.float16 else 2.0**-8
    tol = half_ulp * ref.abs() + 2.0**-18 * R.abs().max().double() * x.abs().sum(-1, keepdim=True) + 2.0**-25
    assert bool(((out - ref).abs() <= tol).all()), float(((out - ref).abs() - tol).max())


# 33, 70: a second, partly filled 32-row tile; 257, 300: a second item of a workgroup's 256
# rows; (2, 8, 8200): more items than the grid's 4096 waves, 8200 % 32 rows left in the last item
@pytest.mark.parametrize("shape", [(1, 1, 1, 128), (2, 3, 33, 128), (1, 2, 70, 128), (1, 3, 257, 128), (2, 8, 8200, 128)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [4, 3, 2])
def test_rotate_dequant(dev, bits, dtype, shape):
    print(f"case rotate_dequant bits={bits} dtype={dtype} shape={shape}", flush=True)
    R = frq._random_orthogonal(128).to(dev)
    for axis in (_lib.AXIS_CHANNEL, _lib.AXIS_TOKEN):
        packed, scale = _inputs(shape, bits, axis, dtype, dev)
        _check(packed, scale, R, bits, dtype)
        _check(packed, scale, R * 300.0, bits, dtype)  # entries far above and below an orthogonal matrix's
        _check(packed, scale * 64.0, R * 1e-4, bits, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("bits", [4, 3, 2])
@pytest.mark.parametrize("size", [2.0**-4, 1.0, 2.0**20])  # 2^-4: a scale of 2^14, the careful branch in fp16
def test_rotate_dequant_last_bits_of_R(dev, bits, dtype, size):
    """The difference of two rows of R that agree in 21 bits is exact in float32: all 24 bits count."""
    g = torch.Generator().manual_seed(8)
    w = torch.rand(128, generator=g) + 1.0
    R = torch.zeros(128, 128)
    R[17], R[90] = w, (w.view(torch.int32) & ~7).view(torch.float32)
    R[3] = torch.rand(128, generator=g)
    R = (R * size).to(dev)
    codes = torch.zeros(1, 1, 70, 128, dtype=torch.int8, device=dev)
    codes[..., 17], codes[..., 90] = 1, -1
    packed = codes if bits == 3 else frq._pack_codes(codes, bits)
    scale = torch.full((1, 1, 70, 1), 2.0**10 / size, dtype=dtype, device=dev)
    out = frq.rotated_dequant_v(packed, scale, R, bits, dtype)
    want = ((R[17].double() - R[90].double()) * scale.double().flatten()[0]).to(dtype)
    assert int((want != 0).sum()) > 64
    assert torch.equal(out, want.expand_as(out))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_rotate_dequant_layouts(dev, dtype):
    """Strided and 16-byte-unaligned codes, an unaligned and a transposed R, a float32 scale."""
    packed, scale = _inputs((2, 2, 90, 128), 4, _lib.AXIS_CHANNEL, dtype, dev)
    R = frq._random_orthogonal(128).to(dev)
    want = frq.rotated_dequant_k(packed, scale, R, 4, dtype)
    wide = torch.zeros(2, 2, 95, 64, dtype=torch.uint8, device=dev)
    wide[:, :, 3:93] = packed
    assert torch.equal(frq.rotated_dequant_k(wide[:, :, 3:93], scale, R, 4, dtype), want)
    flat = torch.zeros(packed.numel() + 4, dtype=torch.uint8, device=dev)
    flat[4:] = packed.reshape(-1)
    assert torch.equal(frq.rotated_dequant_k(flat[4:].view(packed.shape), scale.float(), R, 4, dtype), want)
    rf = torch.zeros(128 * 128 + 1, device=dev)
    rf[1:] = R.reshape(-1)
    assert torch.equal(frq.rotated_dequant_k(packed, scale, rf[1:].view(128, 128), 4, dtype), want)
    assert torch.equal(frq.rotated_dequant_k(packed, scale, R.T.contiguous().T, 4, dtype), want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("axis", [_lib.AXIS_CHANNEL, _lib.AXIS_TOKEN])
def test_rotate_dequant_non_finite(dev, axis, dtype):
    """inf, NaN and overflowing scales give inf and NaN where the two-step path does."""
    packed, scale = _inputs((1, 2, 40, 128), 4, axis, dtype, dev)
    packed[:, :, 5] = 0x17  # no zero codes in row 5, some elsewhere
    s = scale.view(2, -1)
    s[0, 5], s[1, 7], s[0, 9] = float("inf"), float("nan"), 6.0e4
    R = frq._random_orthogonal(128).to(dev)
    out = frq.rotated_dequant_k(packed, scale, R, 4, dtype).float()
    x = dequant_sym(packed, scale, 4, dtype)
    ref = (x.float() @ R).to(dtype).float()
    assert torch.equal(out.isnan(), ref.isnan())
    assert torch.equal(out.isposinf(), ref.isposinf()) and torch.equal(out.isneginf(), ref.isneginf())
    fin = ref.isfinite()
    tol = 2.0**-7 * ref.abs() + 2.0**-18 * x.float().nan_to_num(0, 0, 0).abs().sum(-1, keepdim=True)
    assert bool(((out - ref).abs() <= tol)[fin].all())


def test_rotate_dequant_gradient_of_R(dev):
    """A rotation that records gradients keeps the differentiable path."""
    packed, scale = _inputs((1, 1, 20, 128), 4, _lib.AXIS_TOKEN, torch.float16, dev)
    R = frq._random_orthogonal(128).to(dev).requires_grad_()
    frq.rotated_dequant_v(packed, scale, R, 4, torch.float16).float().sum().backward()
    assert R.grad is not None and bool(R.grad.isfinite().all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("axis", [_lib.AXIS_CHANNEL, _lib.AXIS_TOKEN])
@pytest.mark.parametrize("what", ["inf", "nan", "large", "largest"])
def test_rotate_dequant_extreme_R(dev, axis, dtype, what):
    """Entries of R that are no piece of 16 bits (inf, NaN, a float32 that rounds to a 16-bit inf)
    or far from 1: inf, NaN and finite values where the 64-bit product's rounding has them."""
    packed, scale = _inputs((1, 2, 40, 128), 4, axis, dtype, dev)
    R = frq._random_orthogonal(128).to(dev)
    if what == "inf":
        R[5, 9], R[77, 20], R[78, 20], R[3, 127] = float("inf"), float("inf"), -float("inf"), -float("inf")
    elif what == "nan":
        R[5, 9] = float("nan")
    elif what == "large":
        R = R * 1e25
    else:
        R, scale = torch.zeros_like(R), scale * 2.0**-9
        R[4, 4], R[6, 7] = 3.4e38, -3.4e38
    out = frq.rotated_dequant_k(packed, scale, R, 4, dtype).double()
    x = dequant_sym(packed, scale, 4, dtype).double()
    ref = torch.where(x.unsqueeze(-1) == 0, torch.where(R.isfinite(), 0.0, float("nan")).double(), x.unsqueeze(-1) * R.double()).sum(-2)
    rounded = ref.to(dtype).double()
    assert torch.equal(out.isnan(), rounded.isnan())
    assert torch.equal(out.isposinf(), rounded.isposinf()) and torch.equal(out.isneginf(), rounded.isneginf())
    fin = rounded.isfinite()
    tol = (2.0**-10 if dtype == torch.float16 else 2.0**-7) * ref.abs() + 2.0**-18 * R.abs().nan_to_num(0, 0).max().double() * x.abs().sum(-1, keepdim=True)
    assert bool(((out - ref).abs() <= tol)[fin].all())
