"""The packed decode's automatic split count, read from the workspace it asks for.

Fewer splits than fill the GPU are taken only where every wave still holds one
tile (its tiles share the maximum that the 16-bit probabilities are rounded
against); without a GPU the library plans for 256 workgroup slots."""

from __future__ import annotations

import ctypes

import pytest
import torch

from fade_amd import _lib

FMTS = {  # format, bits of K and V, wavefronts of a workgroup
    "int4": (_lib.MID_SYM, 4, 4, 4),
    "sym2": (_lib.MID_SYM, 2, 2, 8),
    "rot4": (_lib.MID_SYM, 4, 4, 4),
    "rot2": (_lib.MID_SYM, 2, 2, 8),
    "asym42": (_lib.MID_ASYM, 4, 2, 8),
    "k4v2": (_lib.MID_K4V2G, 4, 8, 6),
}


def splits(B, Hq, Hkv, S, fmt, sink=4, recent=64, n_splits=0) -> int:
    """The split count of a call of S middle tokens (addresses are only checked for alignment)."""
    a = _lib.DecodeArgs()
    a.B, a.Hq, a.Hkv, a.D = B, Hq, Hkv, 128
    a.q = a.out = 1 << 20
    a.q_sb, a.q_sh = Hq * 128, 128
    a.sm_scale, a.n_splits = 0.1, n_splits
    for t, n in ((a.sink, sink), (a.recent, recent)):
        t.k = t.v = 1 << 20
        t.len, t.k_sb, t.k_sh, t.k_ss, t.v_sb, t.v_sh, t.v_ss = n, 1 << 20, 1 << 10, 128, 1 << 20, 1 << 10, 128
    m = a.mid
    m.fmt, m.k_bits, m.v_bits, _ = FMTS[fmt]
    m.group, m.len, m.v_rows = (32 if fmt == "asym42" else 64), S, -(-S // 64) * 64
    m.k_codes = m.v_codes = m.k_scale = m.v_scale = m.k_zero = m.v_zero = 1 << 20
    a.rotation = 1 << 20 if fmt.startswith("rot") else None
    nb = ctypes.c_int64(0)
    _lib.check(_lib.load().fade_tiered_decode_workspace_bytes(ctypes.byref(a), nb), "workspace")
    passes = (Hq // Hkv + 3) // 4
    r256 = lambda x: -(-x // 256) * 256  # noqa: E731
    rows = B * max(Hq, 4 * Hkv * passes)
    for n in range(1, 65536):
        if r256(4 * B * Hkv * passes) + r256(8 * rows * n) + 512 * rows * n == nb.value:
            return n
    raise AssertionError(nb.value)


@pytest.mark.skipif(torch.cuda.is_available(), reason="plans for the GPU that is there")
@pytest.mark.parametrize("fmt", list(FMTS))
@pytest.mark.parametrize("B,Hq,Hkv", [(1, 32, 8), (1, 4, 1), (4, 32, 8), (16, 32, 8)])
def test_fewer_splits_only_of_one_tile_per_wave(B, Hq, Hkv, fmt):
    waves, slots, rot = FMTS[fmt][3], 256, fmt.startswith("rot")
    most = (slots + B * Hkv // 2) // (B * Hkv)
    fewer = 0
    for S in (1, 64, 65, 200, 400, 700, 1030, 2048, 4099, 9000, 16384, 32000):
        tiles = -(-S // 64) + (0 if rot else -(-68 // 16))
        cap = max(1, min(most - rot, tiles))
        per = -(-tiles // cap)
        n = splits(B, Hq, Hkv, S, fmt) - rot
        if per > waves:
            assert n == -(-tiles // per), S
        else:
            assert -(-tiles // waves) <= n <= cap and -(-tiles // n) <= waves, S
            fewer += n < cap
    assert fewer > 0 or B == 16


def test_forced_split_counts_are_taken():
    for n in (1, 2, 3, 7):
        assert splits(1, 32, 8, 64 * 42 - 320, "int4", n_splits=n) == n
