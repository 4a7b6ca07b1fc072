"""Per-channel INT4 quantizer in one pass (a (b, h)'s workgroups exchange their column
maxima) and its bounded wait, against the reference's op sequence on the CPU, bit for bit."""

from __future__ import annotations

import pytest
import torch

from fade_amd import _lib
from fade_amd import quant as fq

pytestmark = pytest.mark.gpu


def _reference(k):
    """fade/quant.py:61-75 with torch's per-op rounding; NaN products give code 0."""
    absmax = k.abs().amax(dim=-2, keepdim=True).clamp(min=1e-8)
    q = (k * (7 / absmax)).round().clamp(-8, 7).nan_to_num(0.0).to(torch.int32)
    return ((q[..., 0::2] & 15) << 4 | (q[..., 1::2] & 15)).to(torch.uint8), absmax / 7


def _with_polls(k, polls):
    B, H, S, D = k.shape
    packed = torch.empty(B, H, S, D // 2, dtype=torch.uint8, device=k.device)
    scale = torch.empty(B, H, 1, D, dtype=k.dtype, device=k.device)
    nb = fq.ctypes_i64()
    _lib.check(_lib.load().fade_quant_k_int4_workspace_bytes(B, H, S, D, nb), "ws")
    ws = torch.full((nb.value,), 255, dtype=torch.uint8, device=k.device)  # contents arbitrary
    _lib.call("fade_quant_k_int4_polls", k.data_ptr(), _lib.DTYPE_CODES[k.dtype], B, H, S, D, *k.stride()[:3], polls,
              packed.data_ptr(), scale.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream_of(k))
    return packed, scale


# one workgroup per slice; two, the second with one row; a slice's last rows partly filled;
# 64 slices with 16 rows per thread; more workgroups than may wait (two passes); the other
# instances' head dims
SHAPES = [(1, 2, 5, 128), (1, 3, 65, 128), (2, 2, 700, 128), (8, 8, 1100, 128), (1, 1, 9000, 128),
          (1, 2, 300, 32), (2, 2, 260, 64), (1, 2, 200, 256), (3, 1, 333, 96)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_quant_k_int4_single_pass(dev, shape, dtype):
    print(f"case quant_k_int4 single pass {shape} {dtype}", flush=True)
    g = torch.Generator().manual_seed(sum(shape))
    B, H, S, D = shape
    k = (torch.randn(B, H, S + 3, D, generator=g) * torch.exp(0.5 * torch.randn(D, generator=g))).to(dtype)
    k[:, :, S // 2, :] *= 3  # every column's maximum in one workgroup's rows
    k[..., 3], k[..., 5] = 0, 1e-7
    k[0, 0, 1, 2], k[0, 0, 2, 4], k[0, 0, S - 1, 6] = float("inf"), float("nan"), -float("inf")
    view = k.to(dev)[:, :, 1 : S + 1]  # strided rows, as the cache's middle slice
    want, scale = _reference(k[:, :, 1 : S + 1])
    for polls in (None, 0, 1 << 20):
        p, s = fq.quant_k_int4(view) if polls is None else _with_polls(view, polls)
        assert torch.equal(p.cpu(), want), polls
        assert torch.equal(s.cpu().nan_to_num(-1.0), scale.nan_to_num(-1.0)), polls


def test_quant_k_int4_two_streams(dev):
    """Overlapping calls on two streams do not share an exchange area."""
    g = torch.Generator().manual_seed(1)
    ks = [torch.randn(4, 8, 2000, 128, generator=g).half().to(dev) for _ in range(2)]
    want = [_reference(k.cpu())[0] for k in ks]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    out = [[], []]
    for _ in range(8):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                out[i].append(fq.quant_k_int4(ks[i])[0])
    torch.cuda.synchronize()
    assert all(torch.equal(p.cpu(), want[i]) for i in (0, 1) for p in out[i])


def test_quant_k_int4_captured(dev):
    """A captured call replays: every replay equals the eager result."""
    g = torch.Generator().manual_seed(2)
    k = torch.randn(2, 4, 1500, 128, generator=g).half().to(dev)
    fq.quant_k_int4(k)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        p, s = fq.quant_k_int4(k)
    for r in range(4):
        k.copy_(torch.randn(2, 4, 1500, 128, generator=g).half())
        graph.replay()
        torch.cuda.synchronize()
        pe, se = fq.quant_k_int4(k)
        assert torch.equal(p, pe) and torch.equal(s, se), r
        assert torch.equal(pe.cpu(), _reference(k.cpu())[0])
