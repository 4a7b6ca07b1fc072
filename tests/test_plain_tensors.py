"""``_lib.plain``: whether a kernel may stand in for tensor ops, which a tracer would have recorded."""

from __future__ import annotations

import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode

from fade_amd import _lib


class _Mode(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_plain():
    x = torch.ones(3)
    assert _lib.plain(x, torch.nn.Parameter(x, requires_grad=False))
    assert not _lib.plain(x.clone().requires_grad_())
    with torch.no_grad():
        assert _lib.plain(x.clone().requires_grad_())


def test_not_plain_while_something_records():
    seen = {}

    def f(name):
        def g(x):
            seen[name] = _lib.plain(x)
            return x + 1

        return g

    x = torch.ones(3)
    torch.jit.trace(f("jit"), x, check_trace=False)
    make_fx(f("make_fx"))(x)
    make_fx(f("make_fx fake"), tracing_mode="fake")(x)
    with _Mode():
        f("dispatch mode")(x)
    torch.func.vmap(f("vmap"))(x)
    torch.func.grad(lambda y: f("grad")(y).sum())(x)
    torch.func.jvp(f("jvp"), (x,), (x,))
    assert seen == dict.fromkeys(seen, False) and len(seen) == 7
    assert _lib.plain(x)


def test_not_plain_where_memory_is_not_the_value():
    assert not _lib.plain(torch.ones(4, dtype=torch.complex64).conj().imag)
    assert not _lib.plain(torch.ones(4, dtype=torch.complex64).conj())
