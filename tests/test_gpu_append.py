"""``TieredKVCache.update``'s append in one launch (``fade_append_rows``) against tensor copies."""

from __future__ import annotations

import pytest
import torch

from fade_amd import cache as fc

pytestmark = pytest.mark.gpu


def _buffers(B, H, cap, D, dtype, dev):
    z = lambda *s, **k: torch.full(s, -1, device=dev, **k)  # noqa: E731
    return z(B, H, cap, D, dtype=dtype), z(B, H, cap, D, dtype=dtype), z(cap, dtype=torch.long)


# one row; rows past a block's 256 units; 16-byte rows; a head_dim that is no power of two
@pytest.mark.parametrize("B,H,n,D,at,cap", [(2, 4, 1, 128, 127, 128), (1, 2, 300, 128, 3, 400), (3, 1, 5, 8, 0, 5), (2, 3, 17, 80, 9, 64),
                                            (1, 1, 2100, 256, 1, 2101)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_append_rows(dev, B, H, n, D, at, cap, dtype):
    g = torch.Generator().manual_seed(n)
    k = torch.randn(B, n, H, D, generator=g).to(dtype).to(dev).transpose(1, 2)  # as a projection's heads come
    v = torch.randn(B, H, n + 2, D, generator=g).to(dtype).to(dev)[:, :, 2:]
    bk, bv, bp = _buffers(B, H, cap, D, dtype, dev)
    want = [t.clone() for t in (bk, bv, bp)]
    want[0][:, :, at : at + n], want[1][:, :, at : at + n] = k, v
    want[2][at : at + n] = torch.arange(70, 70 + n, device=dev)
    assert fc._append_rows(k, v, bk, bv, bp, at, 70)
    assert all(torch.equal(a, b) for a, b in zip((bk, bv, bp), want))


def test_append_rows_left_to_tensor_ops(dev):
    """Calls the kernel does not take, and the cache's result for them."""
    r = lambda *s, dt=torch.float16: torch.randn(*s, device=dev).to(dt)  # noqa: E731
    cases = {
        "unaligned": (r(1, 2, 3, 129)[..., 1:], r(1, 2, 3, 128)),
        "short rows": (r(1, 2, 3, 12), r(1, 2, 3, 12)),
        "strided rows": (r(1, 2, 128, 3).transpose(2, 3), r(1, 2, 3, 128)),
        "double": (r(1, 2, 3, 128, dt=torch.float64), r(1, 2, 3, 128, dt=torch.float64)),
        "mixed": (r(1, 2, 3, 128), r(1, 2, 3, 128, dt=torch.float32)),
        "gradient": (r(1, 2, 3, 128).requires_grad_(), r(1, 2, 3, 128)),
    }
    for name, (k, v) in cases.items():
        bk = torch.zeros(1, 2, 8, k.shape[-1], dtype=k.dtype, device=dev)
        assert not fc._append_rows(k, v, bk, torch.zeros_like(bk), torch.zeros(8, dtype=torch.long, device=dev), 0, 0), name
        if name in ("double", "mixed"):
            continue
        c = fc.TieredKVCache(n_sink=2, recent_window=4, head_dim=int(k.shape[-1]))
        c.update(k, v, 0)
        ko, vo = c.update(k, v, 0)
        assert torch.equal(ko, torch.cat([k, k], -2)) and torch.equal(vo, torch.cat([v, v], -2)), name
        assert c._layers[0].fp16_pos.tolist() == list(range(6))
    k, v = cases["gradient"]
    c = fc.TieredKVCache(n_sink=2, recent_window=4, head_dim=128)
    c.update(k, v, 0)[0].float().sum().backward()
    assert torch.equal(k.grad, torch.ones_like(k))


def test_append_grows_and_counts_positions(dev):
    c = fc.TieredKVCache(n_sink=2, recent_window=4, head_dim=64)
    parts = [torch.randn(2, 3, n, 64, device=dev).half() for n in (100, 27, 1, 1, 200, 0, 1)]
    for t in parts:
        ko, vo = c.update(t, -t, 0)
    full = torch.cat(parts, -2)
    assert torch.equal(ko, full) and torch.equal(vo, -full)
    assert c._layers[0].fp16_pos.tolist() == list(range(330))


# no rows of K or V to copy: the positions are appended all the same
@pytest.mark.parametrize("B,H,D", [(0, 2, 64), (2, 0, 64), (2, 3, 0)])
def test_append_of_an_empty_batch(dev, B, H, D):
    k = torch.zeros(B, H, 5, D, device=dev).half()
    bk, bv, bp = _buffers(B, H, 9, D, torch.float16, dev)
    if not fc._append_rows(k, k, bk, bv, bp, 2, 70):  # left to the tensor ops
        return
    assert bp.tolist() == [-1, -1, 70, 71, 72, 73, 74, -1, -1]


def test_update_with_an_empty_batch(dev):
    c = fc.TieredKVCache(n_sink=2, recent_window=4, head_dim=64)
    torch.full((1 << 12,), 77, dtype=torch.long, device=dev)  # freed: what an unwritten buffer may hold
    for n in (300, 1, 1):
        t = torch.zeros(0, 3, n, 64, device=dev).half()
        assert c.update(t, t, 0)[0].shape[0] == 0
    assert c._layers[0].fp16_pos.tolist() == list(range(302))


def test_append_counts_as_an_inplace_write(dev):
    """What autograd refused of the copies it refuses of the kernel: a backward over tiers that were
    appended to since, and writes to inference tensors outside inference mode."""
    r = lambda n: torch.randn(1, 2, n, 64, device=dev).half()  # noqa: E731
    c = fc.TieredKVCache(n_sink=2, recent_window=4, head_dim=64)
    c.update(r(5), r(5), 0)
    w = r(5).requires_grad_()
    out = (w * c._layers[0].fp16_k).sum()
    c.update(r(1), r(1), 0)
    with pytest.raises(RuntimeError, match="inplace operation"):
        out.backward()
    with torch.inference_mode():
        c = fc.TieredKVCache(n_sink=2, recent_window=4, head_dim=64)
        c.update(r(5), r(5), 0)
        c.update(r(1), r(1), 0)
    with pytest.raises(RuntimeError, match="[Ii]nference"):
        c.update(r(1), r(1), 0)


def test_append_off_the_current_device(dev, monkeypatch):
    """Tensors of another device than the current one, on whose streams a launch would go, take the copies."""
    k = torch.randn(1, 2, 3, 64, device=dev).half()
    bk, bv, bp = _buffers(1, 2, 8, 64, torch.float16, dev)
    assert fc._append_rows(k, k, bk, bv, bp, 0, 0)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert not fc._append_rows(k, k, bk, bv, bp, 3, 3)
