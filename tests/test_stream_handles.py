"""Memory handed to a raw stream handle: the default stream's handle is 0, which
``torch.cuda.ExternalStream`` takes as "none given" (it returns another stream)."""

from __future__ import annotations

import contextlib

import pytest
import torch

from fade_amd import _lib


@pytest.fixture
def streams(monkeypatch):
    """torch's stream calls without a GPU: the stream that is current when memory is made."""
    seen = []
    current = []

    @contextlib.contextmanager
    def use(stream):
        current.append(stream)
        yield
        current.pop()

    def made(n, **kw):
        seen.append(current[-1] if current else "current")
        return torch.ones(n, dtype=torch.uint8).fill_(0)

    monkeypatch.setattr(torch.cuda, "ExternalStream", lambda h, device=None: ("external", h) if h else ("pool", 0))
    monkeypatch.setattr(torch.cuda, "default_stream", lambda device=None: ("default", device.index))
    monkeypatch.setattr(torch.cuda, "stream", use)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(_lib.torch, "zeros", made)
    monkeypatch.setattr(_lib.torch, "empty", made)
    monkeypatch.setattr(_lib, "_STREAM_WS", {})
    return seen


def test_decode_workspace_is_zeroed_on_its_stream(streams):
    dev = torch.device("cuda", 3)
    _lib.stream_workspace(100, dev, 0, 8)
    _lib.stream_workspace(100, dev, 0, 8)  # the same buffer
    _lib.stream_workspace(100, dev, 0x1234, 8)
    assert streams == [("default", 3), ("external", 0x1234)]


def test_prefill_sums_live_on_the_stream_of_the_run(streams):
    from fade_amd.kernels.prefill import TieredPrefillPlan

    plan = object.__new__(TieredPrefillPlan)
    plan.out, plan.workspace, plan._ws_stream, plan._argp = torch.full((1,), 0), torch.full((64,), 0, dtype=torch.uint8), 0x55, None
    calls = []
    plan._fn = lambda argp, ws, n, stream: calls.append((ws == plan.workspace.data_ptr(), n, stream)) or 0
    plan.run(0x55)  # the plan's own
    plan.run(0)
    plan.run(0x77)
    assert calls == [(True, 64, 0x55), (False, 64, 0), (False, 64, 0x77)]
    assert streams == [("default", None), ("external", 0x77)]
