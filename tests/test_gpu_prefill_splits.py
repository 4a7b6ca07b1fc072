"""Chunk prefill with its keys split over workgroups (calls too small to fill the GPU),
against a 64-bit softmax and against the unsplit kernel."""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

from fade_amd import _lib
from fade_amd.kernels import MiddleTier
from fade_amd.kernels.prefill import TieredPrefillPlan
from fade_amd.quant import dequant_int4, quant_k_int4, quant_v_int4

pytestmark = pytest.mark.gpu


def _plan(dev, B, Hq, Hkv, D, Sq, rows, dtype, mask, seed=5):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)  # noqa: E731
    caps = [max(r[i] for r in rows) for i in range(3)]
    kv = [(rnd(B, Hkv, c, D), rnd(B, Hkv, c, D)) for c in caps]
    mid = None
    if caps[1]:
        (kq, ks), (vq, vs) = quant_k_int4(kv[1][0]), quant_v_int4(kv[1][1])
        mid = MiddleTier("int4", kq, vq, ks, vs)
    chunk = (rnd(B, Hkv, Sq, D), rnd(B, Hkv, Sq, D))
    q = rnd(B, Hq, Sq, D)
    lens = torch.tensor(rows, dtype=torch.int32)
    return TieredPrefillPlan(q, chunk, kv[0] if caps[0] else None, mid, kv[2] if caps[2] else None, lens=lens, mask=mask)


def _unsplit(plan):
    out = torch.empty_like(plan.out)
    keep, plan.args.out = plan.args.out, out.data_ptr()
    s = torch.cuda.current_stream(out.device).cuda_stream
    _lib.check(_lib.load().fade_tiered_prefill_attn(ctypes.byref(plan.args), s), "unsplit")
    plan.args.out = keep
    return out


def _exact(plan, mask):
    q, chunk, sink, mid, rec, lens = plan._keep[:6]
    B, Hq, Sq, D = q.shape
    G = Hq // chunk[0].shape[1]
    out = torch.empty(B, Hq, Sq, D, dtype=torch.float64, device=q.device)
    deq = None if mid is None else (dequant_int4(mid.k_codes, mid.k_scale, q.dtype), dequant_int4(mid.v_codes, mid.v_scale, q.dtype))
    for b in range(B):
        n = lens[b].tolist()
        parts = [(t, m) for t, m in zip((sink, deq, rec, chunk), (*n, Sq)) if t is not None]
        k, v = (torch.cat([t[i][b, :, :m].double() for t, m in parts], dim=-2).repeat_interleave(G, 0) for i in (0, 1))
        S, j = k.shape[1], torch.arange(Sq, device=q.device)
        last = j + (S - Sq if mask == "bottom_right" else 0) if mask != "none" else torch.full_like(j, S)
        s = (q[b].double() @ k.transpose(-1, -2).contiguous()) / math.sqrt(D)
        s.masked_fill_(torch.arange(S, device=q.device)[None, None, :] > last[None, :, None], -math.inf)
        out[b] = torch.softmax(s, -1) @ v
    return out


@pytest.mark.parametrize(
    "B,Hq,Hkv,D,Sq,rows",
    [
        (1, 4, 1, 128, 16, [(4, 1000, 64)]),  # one row, one 32-query block
        (1, 14, 2, 64, 70, [(4, 2999, 61)]),  # two head passes, two groups, a partial last block
        (3, 8, 2, 128, 40, [(4, 1500, 64), (0, 30, 5), (4, 0, 1)]),  # splits past a short row's tiles
        (2, 16, 8, 256, 33, [(4, 700, 20), (1, 513, 64)]),  # one wave per SIMD
        (1, 4, 4, 32, 130, [(0, 900, 0)]),  # MHA: a group's waves cover four query blocks
        (1, 8, 2, 96, 20, [(4, 640, 3)]),  # head_dim below its instance's capacity
        (1, 2, 1, 40, 9, [(600, 0, 200)]),  # no middle tier; 10 threads per merged row
    ],
)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("mask", ["bottom_right", "top_left", "none"])
def test_prefill_key_splits(dev, B, Hq, Hkv, D, Sq, rows, dtype, mask):
    print(f"case prefill splits B={B} Hq={Hq} Hkv={Hkv} D={D} Sq={Sq} rows={rows} {dtype} {mask}", flush=True)
    plan = _plan(dev, B, Hq, Hkv, D, Sq, rows, dtype, mask)
    assert plan.workspace is not None  # the call is split
    out = plan.run().double()
    ref, one = _exact(plan, mask), _unsplit(plan).double()
    # the suite's bars for this kernel; the split may not be further off than the unsplit
    # kernel by more than the rounding of one output
    eps = 2.0**-11 if dtype == torch.float16 else 2.0**-8
    err, err1 = (out - ref).abs(), (one - ref).abs()
    bar = 2e-3 if dtype == torch.float16 else 4e-3
    assert bool((err <= bar + (0 if dtype == torch.float16 else 2.0**-7) * ref.abs()).all()), float(err.max())
    assert float(err.pow(2).mean().sqrt()) <= float(err1.pow(2).mean().sqrt()) * 1.1 + eps * 1e-2
    assert torch.equal(plan.run().double(), out)  # merged in a fixed order


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("what", ["K nan", "K inf", "K -inf scores", "V nan", "V inf", "V both infs"])
def test_prefill_split_non_finite(dev, dtype, what):
    """inf and NaN in one split's keys reach the merged rows as they reach the unsplit kernel's."""
    plan = _plan(dev, 2, 4, 2, 128, 40, [(4, 1500, 64), (4, 700, 64)], dtype, "bottom_right")
    assert plan.workspace is not None
    q, chunk, sink, mid, rec = plan._keep[:5]
    inf = float("inf")
    if what == "K nan":
        rec[0][0, 1, 7, 5] = float("nan")
    elif what == "K inf":
        rec[0][0, 1, 7, 5] = inf
    elif what == "K -inf scores":  # a key that no query of the group sees
        q[0, 2:, :, 5] = q[0, 2:, :, 5].abs() + 1
        rec[0][0, 1, 7, 5] = -inf
    elif what == "V nan":
        sink[1][0, 1, 2, 9] = float("nan")
    elif what == "V inf":
        sink[1][0, 1, 2, 9] = -inf
    else:  # +inf and -inf in different splits
        sink[1][0, 1, 2, 9], rec[1][0, 1, 7, 9] = inf, -inf
    out, one = plan.run().float(), _unsplit(plan).float()
    assert torch.equal(out.isnan(), one.isnan()) and torch.equal(out.isposinf(), one.isposinf()) and torch.equal(out.isneginf(), one.isneginf())
    assert bool(out[1].isfinite().all() and out[0, :2].isfinite().all())
    assert bool(out.isfinite().all()) == (what == "K -inf scores")
    fin = out.isfinite()
    assert bool(((out - one).abs() <= (2e-3 if dtype == torch.float16 else 8e-3) + 2.0**-7 * one.abs())[fin].all())


def test_prefill_split_workspace_checked(dev):
    plan = _plan(dev, 1, 4, 1, 128, 16, [(4, 1000, 64)], torch.float16, "bottom_right")
    lib, s = _lib.load(), torch.cuda.current_stream().cuda_stream
    need = plan.workspace.numel()
    assert lib.fade_tiered_prefill_attn_ws(ctypes.byref(plan.args), None, 0, s) == _lib.FADE_EINVAL
    assert lib.fade_tiered_prefill_attn_ws(ctypes.byref(plan.args), plan.workspace.data_ptr(), need - 1, s) == _lib.FADE_EINVAL


def test_prefill_split_on_another_stream(dev):
    """Plans made on one stream, run on another and dropped at once: their sums are not overwritten."""
    plan = _plan(dev, 1, 4, 1, 128, 16, [(4, 1000, 64)], torch.float16, "bottom_right")
    want = plan.run().clone()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    outs = []
    for _ in range(20):
        p = TieredPrefillPlan(*plan._keep[:5], lens=plan._keep[5])
        outs.append(p.run(side.cuda_stream))
        del p
        torch.full((1 << 20,), 255, dtype=torch.uint8, device=dev)
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs)


def test_prefill_split_on_the_default_stream(dev):
    """A plan made on a side stream, run on the default stream and dropped at once: what is
    allocated on the side stream next does not overwrite its sums."""
    plan = _plan(dev, 1, 4, 1, 128, 16, [(4, 1000, 64)], torch.float16, "bottom_right")
    want, args = plan.run().clone(), plan._keep
    side, busy = torch.cuda.Stream(), torch.randn(4096, 4096, device=dev)
    torch.cuda.synchronize()
    outs = []
    for _ in range(10):
        with torch.cuda.stream(side):
            p = TieredPrefillPlan(*args[:5], lens=args[5])
        torch.cuda.current_stream().wait_stream(side)
        busy @ busy  # the run starts after the fill below would
        outs.append(p.run())
        n = p.workspace.numel()
        outs[-1].record_stream(torch.cuda.current_stream())
        del p
        with torch.cuda.stream(side):
            torch.full((n,), 255, dtype=torch.uint8, device=dev)
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs)


def test_prefill_split_captured(dev):
    """A captured split call replays to the eager result."""
    plan = _plan(dev, 1, 14, 2, 64, 70, [(4, 2000, 61)], torch.float16, "bottom_right")
    want = plan.run().clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.run()
    for _ in range(3):
        plan.out.zero_()
        plan.workspace.fill_(255)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(plan.out, want)
