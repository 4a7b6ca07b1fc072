"""Workloads of the tiered KV cache that are timed: what a program does with one layer.

Five kinds of work, each through the entry point that a serving program calls:

  decode      one query token per row over [sink | packed middle | recent]: a
              ``TieredDecodePlan`` bound once and run for every token
  prefill     a chunk of queries per row over the same tiers plus the chunk's
              own keys: a ``TieredPrefillPlan``
  compress    a layer's middle K and V into the packed format of a quantization
              backend, at a tier reassignment
  decompress  the packed middle back to floats, for a model that attends over
              the materialized cache
  layer       a ``TieredKVCache`` layer's life: the prompt's K/V, the
              score-driven reassignment, then decode steps

Inputs follow the benchmark's distributions: K ~ N(0, 1) with per-channel
scales ~ LogNormal(0, 0.5), V and Q ~ N(0, 1), scores ~ Exponential(1).
"""

from __future__ import annotations

import math

import torch

from fade_amd.backends import get_backend
from fade_amd.cache import TieredKVCache
from fade_amd.kernels.prefill import TieredPrefillPlan
from fade_amd.kernels.tiered_attn import MiddleTier, TieredDecodePlan
from fade_amd.policy import reassign_tiers_with_scores
from fade_amd.rope import Vanilla

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
# query heads, kv heads, head_dim: 8B-class GQA-4, Qwen2.5-7B's GQA-7, a 70B-class
# GQA-8, Qwen2.5-0.5B's 14/2 at head_dim 64, Gemma's 16/8 at head_dim 256
SHAPES = ((32, 8, 128), (28, 4, 128), (64, 8, 128), (14, 2, 64), (16, 8, 256))
THETA = 1.0e6
# bounds of one case's size: elements of one K or V middle tier, and prefill products
MOST_ELEMENTS = 16 * 8 * 8192 * 128
MOST_PREFILL_FLOPS = 6.0e11


# ------------------------------------------------------------------ the cases
def listed() -> list[dict]:
    return [
        # one chat sequence on a small model: latency and launches are what counts
        dict(name="decode_b1_d64", kind="decode", B=1, Hq=14, Hkv=2, D=64, S=1000, sink=4, recent=64, fmt="int4", dtype="fp16"),
        # the headline workload: an 8B-class layer, a batch of 16 at 8K tokens
        dict(name="decode_b16_8k", kind="decode", B=16, Hq=32, Hkv=8, D=128, S=8192, sink=4, recent=64, fmt="int4", dtype="fp16"),
        # a bfloat16 model with 7 query heads per kv head, a length that fits no tile
        dict(name="decode_bf16_gqa7", kind="decode", B=8, Hq=28, Hkv=4, D=128, S=4099, sink=4, recent=128, fmt="int4", dtype="bf16"),
        # long context, the mixed-precision tier: 4-bit K and 2-bit V in asymmetric groups of 32
        dict(name="decode_32k_k4v2", kind="decode", B=4, Hq=32, Hkv=8, D=128, S=32768, sink=4, recent=256, fmt="asym42", dtype="fp16"),
        # long context, the rotated 2-bit backend
        dict(name="decode_32k_rot2", kind="decode", B=4, Hq=32, Hkv=8, D=128, S=32768, sink=4, recent=256, fmt="rot2", dtype="fp16"),
        # a chunk of 128 tokens for each of 32 sequences of very different lengths
        dict(name="prefill_b32_ragged", kind="prefill", B=32, Hq=32, Hkv=8, D=128, Sq=128, Lmin=512, Lmax=16384, sink=4, recent=64, dtype="fp16"),
        # a follow-up prompt in a chat with a small bfloat16 model: odd chunk, odd length
        dict(name="prefill_b2_d64", kind="prefill", B=2, Hq=14, Hkv=2, D=64, Sq=333, Lmin=2999, Lmax=2999, sink=4, recent=64, dtype="bf16"),
        # the reassignment's quantizers at the headline workload's size
        dict(name="compress_int4_b16_8k", kind="compress", B=16, H=8, D=128, S=8124, fmt="int4", dtype="fp16"),
        # the same on a bfloat16 model at an odd size
        dict(name="compress_int4_bf16", kind="compress", B=3, H=4, D=128, S=5003, fmt="int4", dtype="bf16"),
        # the rotated 2-bit backend's quantizers at long context
        dict(name="compress_rot2_32k", kind="compress", B=4, H=8, D=128, S=32508, fmt="rot2", dtype="fp16"),
        # the rotated 4-bit backend read back, as every step of a model with its own attention does
        dict(name="decompress_rot4", kind="decompress", B=4, H=8, D=128, S=8060, fmt="rot4", dtype="fp16"),
        # a layer from the prompt through eviction (400 middle tokens kept) to the first tokens
        dict(name="layer_evict_b8_4k", kind="layer", B=8, Hq=28, Hkv=4, D=128, S=4096, sink=4, recent=64, budget=400, steps=4, dtype="fp16"),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(("decode", "decode", "decode", "prefill", "compress", "compress", "decompress", "layer"))
    Hq, Hkv, D = rng.choice(SHAPES[:1] * 3 + SHAPES)
    dtype = rng.choice(("fp16", "fp16", "bf16"))
    if kind == "decode":
        fmt = rng.choice(("int4", "int4", "rot4", "rot2", "asym44", "asym42", "k4v2")) if D == 128 else "int4"
        B = _log_int(rng, 1, 16)
        S = _log_int(rng, 512, max(512, min(32768, MOST_ELEMENTS // (B * Hkv * D))))
        return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, D=D, S=S, sink=4, recent=rng.choice((32, 64, 128, 256)), fmt=fmt,
                    dtype="fp16" if fmt.startswith("asym") else dtype)
    if kind == "prefill":
        B, Sq = _log_int(rng, 1, 32), _log_int(rng, 16, 512)
        most = int(MOST_PREFILL_FLOPS / (4.0 * B * Hq * Sq * D))
        Lmax = _log_int(rng, 512, max(512, min(16384, most)))
        return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, D=D, Sq=Sq, Lmin=max(128, Lmax // rng.choice((1, 4, 32))), Lmax=Lmax, sink=4,
                    recent=64, dtype=dtype)
    if kind == "layer":
        B, S = _log_int(rng, 1, 8), _log_int(rng, 512, 4096)
        return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, D=D, S=S, sink=4, recent=rng.choice((32, 64, 128)),
                    budget=rng.choice((-1, 200, 400)), steps=4, dtype="fp16")
    fmt = rng.choice(("int4", "int4", "rot4", "rot2", "asym44", "asym42")) if D == 128 else "int4"
    B = _log_int(rng, 1, 16)
    most = MOST_ELEMENTS if kind == "compress" else MOST_ELEMENTS // 4
    S = _log_int(rng, 400, max(400, min(32508, most // (B * Hkv * D))))
    return dict(kind=kind, B=B, H=Hkv, D=D, S=S, fmt=fmt, dtype="fp16" if fmt.startswith("asym") else dtype)


# ----------------------------------------------------------------- the inputs
class _Inputs:
    """Seeded tensors on the GPU: the same for the same case and seed."""

    def __init__(self, seed: int, dtype: torch.dtype) -> None:
        self.gen = torch.Generator(device=DEV).manual_seed(seed)
        self.dtype = dtype

    def normal(self, *shape) -> torch.Tensor:
        return torch.randn(*shape, generator=self.gen, device=DEV, dtype=torch.float32).to(self.dtype)

    def channels(self, H: int, D: int) -> torch.Tensor:
        return torch.exp(0.5 * torch.randn(1, H, 1, D, generator=self.gen, device=DEV))

    def keys(self, chan: torch.Tensor, B: int, S: int) -> torch.Tensor:
        _, H, _, D = chan.shape
        return (torch.randn(B, H, S, D, generator=self.gen, device=DEV) * chan).to(self.dtype)


def _rotation(D: int) -> torch.Tensor:
    """The rotated backend's seeded orthogonal matrix (Q of a Gaussian's QR, seed 42)."""
    q, _ = torch.linalg.qr(torch.randn(D, D, generator=torch.Generator().manual_seed(42)))
    return q.to(DEV)


def _sym(x: torch.Tensor, bits: int, dim: int):
    """Symmetric codes (as floats) and the scale in x's dtype, one scale per slice along ``dim``."""
    top = 2 ** (bits - 1) - 1
    scale = (x.abs().amax(dim=dim, keepdim=True).clamp_min(1e-6) / top).to(x.dtype)
    return (x / scale).float().round_().clamp_(-top - 1, top), scale


def _pack(codes: torch.Tensor, bits: int) -> torch.Tensor:
    """Codes along the last dim into bytes, the first code in the high bits."""
    per = 8 // bits
    c = codes.to(torch.int16).bitwise_and_((1 << bits) - 1).unflatten(-1, (-1, per))
    out = c[..., 0] << (8 - bits)
    for j in range(1, per):
        out |= c[..., j] << (8 - bits * (j + 1))
    return out.to(torch.uint8)


def _asym(x: torch.Tensor, bits: int, group: int = 32):
    """Per-token groups along the last dim: codes (as floats), scale, zero."""
    g = x.unflatten(-1, (-1, group))
    zero = g.amin(dim=-1)
    scale = ((g.amax(dim=-1).float() - zero.float()) / (2**bits - 1)).clamp_min(1e-6).to(x.dtype)
    codes = ((g.float() - zero.float().unsqueeze(-1)) / scale.float().unsqueeze(-1)).round_().clamp_(0, 2**bits - 1)
    return codes.flatten(-2), scale, zero


def _grouped2(x: torch.Tensor, group: int = 64):
    """2-bit codes (as floats) and a scale per (64 tokens, channel), the tokens padded to whole groups."""
    B, H, S, D = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 0, -S % group)).reshape(B, H, -1, group, D)
    scale = xp.abs().amax(dim=-2, keepdim=True).clamp_min(1e-6)
    codes = (xp / scale).float().round_().clamp_(-2, 1)
    return codes.reshape(B, H, -1, D), scale.squeeze(-2)


def _packed_pair(k: torch.Tensor, v: torch.Tensor, fmt: str):
    """The packed middle tier of ``k`` and ``v``: a ``MiddleTier`` (or its tensors) and the rotation."""
    if fmt == "int4":
        (kc, ks), (vc, vs) = _sym(k, 4, -2), _sym(v, 4, -1)
        return MiddleTier("int4", _pack(kc, 4), _pack(vc, 4), ks, vs), None
    if fmt.startswith("rot"):
        bits, R = int(fmt[3]), _rotation(k.shape[-1])
        (kc, ks), (vc, vs) = _sym((k.float() @ R.T).to(k.dtype), bits, -2), _sym((v.float() @ R.T).to(v.dtype), bits, -1)
        return MiddleTier("sym", _pack(kc, bits), _pack(vc, bits), ks, vs, k_bits=bits, v_bits=bits), R
    if fmt.startswith("asym"):
        kb, vb = int(fmt[4]), int(fmt[5])
        (kc, ks, kz), (vc, vs, vz) = _asym(k, kb), _asym(v, vb)
        return MiddleTier("asym", _pack(kc, kb), _pack(vc, vb), ks, vs, kz, vz, k_bits=kb, v_bits=vb, group=32), None
    (kc, ks), (vc, vs) = _sym(k, 4, -2), _grouped2(v)
    return MiddleTier("k4v2", _pack(kc, 4), vc.to(torch.int8), ks, vs, group=64, length=int(v.shape[2])), None


def _unpack(packed: torch.Tensor, bits: int, signed: bool) -> torch.Tensor:
    per = 8 // bits
    p = packed.to(torch.int16)
    c = torch.stack([(p >> (8 - bits * (j + 1))) & ((1 << bits) - 1) for j in range(per)], dim=-1).flatten(-2)
    return torch.where(c >= 1 << (bits - 1), c - (1 << bits), c) if signed else c


def _mid_in_64(mid: MiddleTier, R, b: int):
    """Row ``b``'s middle K and V in float64, in the model's basis."""
    out = []
    for codes, scale, zero, bits in ((mid.k_codes, mid.k_scale, mid.k_zero, mid.k_bits),
                                     (mid.v_codes, mid.v_scale, mid.v_zero, mid.v_bits)):
        c, s = codes[b], scale[b].double()
        if mid.fmt == "asym":
            x = _unpack(c, bits, False).double().unflatten(-1, (-1, mid.group))
            x = (x * s.unsqueeze(-1) + zero[b].double().unsqueeze(-1)).flatten(-2)
        elif c.dtype == torch.int8:
            x = (c.double() * s.repeat_interleave(mid.group, dim=-2))[:, : mid.length]
        else:
            x = _unpack(c, bits, True).double() * s
        out.append(x if R is None else x @ R.double())
    return out


def _backend(case: dict):
    fmt, D = case["fmt"], case["D"]
    if fmt == "int4":
        return get_backend("int4")
    if fmt.startswith("rot"):
        return get_backend("rotated", head_dim=D, bits=int(fmt[3]))
    return get_backend("asym", head_dim=D, bits=int(fmt[4]), v_bits=int(fmt[5]))


def _attention_inputs(case: dict, seed: int) -> dict:
    """Query, tiers (and the chunk of a prefill) of an attention case."""
    B, Hq, Hkv, D, ns, nr = (case[k] for k in ("B", "Hq", "Hkv", "D", "sink", "recent"))
    i = _Inputs(seed, DTYPES[case["dtype"]])
    chan = i.channels(Hkv, D)
    d = {"sink": (i.keys(chan, B, ns), i.normal(B, Hkv, ns, D)), "recent": (i.keys(chan, B, nr), i.normal(B, Hkv, nr, D))}
    if case["kind"] == "decode":
        n = case["S"] - ns - nr
        d["q"] = i.normal(B, Hq, 1, D)
        d["mid"], d["R"] = _packed_pair(i.keys(chan, B, n), i.normal(B, Hkv, n, D), case["fmt"])
        return d
    Sq = case["Sq"]
    d["q"], d["chunk"] = i.normal(B, Hq, Sq, D), (i.keys(chan, B, Sq), i.normal(B, Hkv, Sq, D))
    lens = torch.randint(case["Lmin"], case["Lmax"] + 1, (B,), generator=torch.Generator().manual_seed(seed))
    lens[0] = case["Lmax"]
    n = lens - ns - nr
    d["mid"], d["R"] = _packed_pair(i.keys(chan, B, int(n.max())), i.normal(B, Hkv, int(n.max()), D), "int4")
    d["lens"] = torch.stack([torch.full((B,), ns), n, torch.full((B,), nr)], dim=1).to(torch.int32)
    return d


def _layer_inputs(case: dict, seed: int) -> dict:
    B, Hq, Hkv, D, S = (case[k] for k in ("B", "Hq", "Hkv", "D", "S"))
    i = _Inputs(seed, DTYPES[case["dtype"]])
    chan = i.channels(Hkv, D)
    g = torch.Generator().manual_seed(seed)
    return {
        "k": i.keys(chan, B, S), "v": i.normal(B, Hkv, S, D),
        "scores": -torch.log(torch.rand(S, generator=g).clamp_min(1e-30)),
        "steps": [(i.normal(B, Hq, 1, D), i.keys(chan, B, 1), i.normal(B, Hkv, 1, D)) for _ in range(case["steps"])],
    }


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "decode":
        d = _attention_inputs(case, seed)
        return {"kind": kind, "plan": TieredDecodePlan(d["q"], d["sink"], d["mid"], d["recent"], rotation=d["R"])}
    if kind == "prefill":
        d = _attention_inputs(case, seed)
        order = torch.argsort(d["lens"][:, 1], descending=True).to(torch.int32)  # the longest rows first
        return {"kind": kind, "plan": TieredPrefillPlan(d["q"], d["chunk"], d["sink"], d["mid"], d["recent"], lens=d["lens"], order=order)}
    if kind == "layer":
        return {"kind": kind, "case": case, **_layer_inputs(case, seed)}
    B, H, D, S = (case[k] for k in ("B", "H", "D", "S"))
    i = _Inputs(seed, DTYPES[case["dtype"]])
    k, v = i.keys(i.channels(H, D), B, S), i.normal(B, H, S, D)
    if kind == "compress":
        return {"kind": kind, "backend": _backend(case), "k": k, "v": v}
    mid, _ = _packed_pair(k, v, case["fmt"])
    ck, cv = {"packed": mid.k_codes, "scale": mid.k_scale}, {"packed": mid.v_codes, "scale": mid.v_scale}
    if mid.k_zero is not None:
        ck["zero"], cv["zero"] = mid.k_zero, mid.v_zero
    return {"kind": kind, "backend": _backend(case), "k": ck, "v": cv, "dtype": DTYPES[case["dtype"]]}


# ------------------------------------------------------------------- one pass
def _run_layer(state: dict) -> dict:
    c = state["case"]
    cache = TieredKVCache(n_sink=c["sink"], recent_window=c["recent"], int4_budget=None if c["budget"] < 0 else c["budget"],
                          dtype=DTYPES[c["dtype"]], head_dim=c["D"], rope_scheme=Vanilla(theta=THETA, head_dim=c["D"]))
    cache.fused = True  # as create_tiered_cache sets it for a model with the "fade" attention
    cache.update(state["k"], state["v"], 0)
    reassign_tiers_with_scores(cache, {0: state["scores"]})
    st = cache._layers[0]
    out = {"sink_k": st.sink_k, "sink_v": st.sink_v, "kq": st.int4_kq, "ks": st.int4_ks, "vq": st.int4_vq, "vs": st.int4_vs}
    for n, (q, k, v) in enumerate(state["steps"]):
        cache.update(k, v, 0)
        out["step%d" % n] = cache.attend(q, 0)
    out["recent_k"], out["recent_v"] = st.fp16_k, st.fp16_v
    return out


def run(state: dict):
    kind = state["kind"]
    if kind in ("decode", "prefill"):
        return state["plan"].run()
    if kind == "layer":
        return _run_layer(state)
    be = state["backend"]
    if kind == "compress":
        return be.compress_k(state["k"]), be.compress_v(state["v"])
    return be.decompress_k(state["k"], state["dtype"]), be.decompress_v(state["v"], state["dtype"])


# --------------------------------------------------------- what a pass has to do
def _bits(fmt: str) -> tuple[int, int]:
    if fmt.startswith("asym"):
        return int(fmt[4]), int(fmt[5])
    if fmt.startswith("rot"):
        return int(fmt[3]), int(fmt[3])
    return 4, 8 if fmt == "k4v2" else 4  # the grouped 2-bit V codes are stored as bytes


def _mid_bytes(fmt: str, n: float, D: int) -> float:
    """Packed K and V of ``n`` tokens of one kv head, with their scales."""
    kb, vb = _bits(fmt)
    if fmt.startswith("asym"):
        meta = n * (D // 32) * 8
    elif fmt == "k4v2":
        meta = 2 * D + -(-n // 64) * D * 2
    else:
        meta = 2 * D + 2 * n
    return n * D * (kb + vb) / 8 + meta


def _kept(case: dict) -> tuple[int, int]:
    """Middle and recent tokens of a layer case after its reassignment."""
    mid = case["S"] - case["sink"] - case["recent"]
    return (mid if case["budget"] < 0 else min(mid, case["budget"])), case["recent"]


def work(case: dict) -> dict:
    kind, B, D = case["kind"], case["B"], case["D"]
    if kind in ("compress", "decompress"):
        n = B * case["H"] * case["S"] * D
        rot = 4.0 * n * D if case["fmt"].startswith("rot") else 0.0
        return {"bytes": 4 * n + B * case["H"] * _mid_bytes(case["fmt"], case["S"], D), "flops": rot}
    Hq, Hkv, ns, nr = case["Hq"], case["Hkv"], case["sink"], case["recent"]
    if kind == "decode":
        n = case["S"] - ns - nr
        nbytes = B * Hkv * ((ns + nr) * D * 4 + _mid_bytes(case["fmt"], n, D)) + 4 * B * Hq * D
        return {"bytes": nbytes, "flops": 4.0 * B * Hq * case["S"] * D}
    if kind == "prefill":
        Sq, L = case["Sq"], 0.5 * (case["Lmin"] + case["Lmax"])  # the mean row
        nbytes = B * Hkv * ((ns + nr + Sq) * D * 4 + _mid_bytes("int4", L - ns - nr, D)) + 4 * B * Hq * Sq * D
        return {"bytes": nbytes, "flops": 4.0 * B * Hq * Sq * D * (L + 0.5 * (Sq + 1))}
    mid, rec = _kept(case)
    tiers = B * Hkv * ((ns + rec) * D * 4 + _mid_bytes("int4", mid, D))
    steps = case["steps"] * (tiers + 4 * B * Hq * D + 8 * B * Hkv * D)
    return {"bytes": 4 * B * Hkv * case["S"] * D + tiers + steps, "flops": 4.0 * case["steps"] * B * Hq * (ns + mid + rec) * D}


def tolerance(case: dict):
    kind, bf16 = case["kind"], case["dtype"] == "bf16"
    if kind in ("compress", "decompress") and not case["fmt"].startswith("rot"):
        return "exact"  # the reference's own rounding, value for value
    if kind == "compress":
        # sums of the rotation in another order move a product across a rounding tie now and then
        return {"rel": 1e-4, "max": 1e-2, "differ": 1e-4}
    if kind == "decompress":
        return {"rel": 1e-2 if bf16 else 1.2e-3}  # 2.7e-4 seen in fp16: x_rot and the result are each rounded once
    # seen against 64 bits: 5e-4 in fp16, 3.3e-3 in bf16 (16-bit probabilities and outputs)
    return {"rel": 1.3e-2 if bf16 else 2.4e-3, "differ": 1e-4}


# ------------------------------------------------------------------- in 64 bits
def _softmax_rows(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, causal: int = 0) -> torch.Tensor:
    """q [Hq, Sq, D] over k, v [Hkv, S, D] in float64; the last ``causal`` keys are the queries' own."""
    Hkv, S, D = k.shape
    q = q.double()
    out = torch.empty_like(q)
    G = q.shape[0] // Hkv
    hide = None
    if causal > 1:
        j = torch.arange(q.shape[1], device=q.device)
        hide = torch.arange(S, device=q.device)[None, :] > (S - causal + j)[:, None]
    for h in range(q.shape[0]):
        s = q[h] @ k[h // G].T / math.sqrt(D)
        if hide is not None:
            s.masked_fill_(hide, -math.inf)
        out[h] = torch.softmax(s, dim=-1) @ v[h // G]
    return out


def _exact_attention(case: dict, seed: int) -> torch.Tensor:
    d = _attention_inputs(case, seed)
    rows = []
    for b in range(case["B"]):
        mk, mv = _mid_in_64(d["mid"], d["R"], b)
        if "lens" in d:
            n = int(d["lens"][b, 1])
            mk, mv = mk[:, :n], mv[:, :n]
        own = d.get("chunk")
        parts = [[t[j][b].double() for t in (d["sink"], d["recent"])] for j in (0, 1)]
        ks, vs = ([parts[j][0], (mk, mv)[j], parts[j][1]] + ([own[j][b].double()] if own else []) for j in (0, 1))
        rows.append(_softmax_rows(d["q"][b], torch.cat(ks, dim=-2), torch.cat(vs, dim=-2), case["Sq"] if own else 0))
    return torch.stack(rows)


def _scales_in_64(x: torch.Tensor, fmt: str, bits: int, dim: int) -> dict:
    x = x.double()
    if fmt.startswith("asym"):
        g = x.unflatten(-1, (-1, 32))
        lo, hi = g.amin(dim=-1), g.amax(dim=-1)
        return {"packed": None, "scale": (hi - lo) / (2**bits - 1), "zero": lo}
    return {"packed": None, "scale": x.abs().amax(dim=dim, keepdim=True) / (2 ** (bits - 1) - 1)}


def _exact_compress(case: dict, seed: int):
    s = prepare(case, seed)
    fmt, (kb, vb) = case["fmt"], _bits(case["fmt"])
    R = _rotation(case["D"]).double() if fmt.startswith("rot") else None
    out = []
    for x, bits, dim in ((s["k"], kb, -2), (s["v"], vb, -1)):
        rows = [_scales_in_64(x[b : b + 1] if R is None else x[b : b + 1].double() @ R.T, fmt, bits, dim) for b in range(case["B"])]
        out.append({f: None if rows[0][f] is None else torch.cat([r[f] for r in rows]) for f in rows[0]})
    return tuple(out)


def _exact_decompress(case: dict, seed: int):
    B, H, D, S = (case[k] for k in ("B", "H", "D", "S"))
    i = _Inputs(seed, DTYPES[case["dtype"]])
    mid, R = _packed_pair(i.keys(i.channels(H, D), B, S), i.normal(B, H, S, D), case["fmt"])
    rows = [_mid_in_64(mid, R, b) for b in range(B)]
    return tuple(torch.stack([r[j] for r in rows]) for j in (0, 1))


def _exact_layer(case: dict, seed: int) -> dict:
    """The tiers and outputs of a layer case, nothing rounded but the packed middle."""
    d = _layer_inputs(case, seed)
    S, D, ns, nr = case["S"], case["D"], case["sink"], case["recent"]
    mid = torch.arange(ns, S - nr)
    if 0 <= case["budget"] < mid.numel():
        mid = mid[torch.argsort(d["scores"][ns : S - nr], descending=True)[: case["budget"]]].sort().values
    keep = torch.cat([torch.arange(ns), mid, torch.arange(S - nr, S)]).to(DEV)
    k, v = d["k"][:, :, keep].double(), d["v"][:, :, keep].double()
    n = int(keep.numel())
    if n < S:  # rotate by (new position - old position)
        freq = THETA ** (-torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D)
        ang = ((torch.arange(n, device=DEV) - keep).double()[:, None] * freq).repeat(1, 2)
        half = torch.cat([-k[..., D // 2 :], k[..., : D // 2]], dim=-1)
        k = k * ang.cos() + half * ang.sin()
    out = {"kq": None, "vq": None, "sink_k": k[:, :, :ns], "sink_v": v[:, :, :ns]}
    m = slice(ns, n - nr)
    hat = []
    for name, x, dim in (("ks", k[:, :, m], -2), ("vs", v[:, :, m], -1)):
        out[name] = x.abs().amax(dim=dim, keepdim=True) / 7
        x = x.half()  # the codes are those of the stored values, by the format's definition: rne(x * (1 / absmax * 7))
        inv = x.abs().amax(dim=dim, keepdim=True).reciprocal() * 7
        hat.append((x * inv).round().clamp(-8, 7).double() * out[name].half().double())
    rec = [k[:, :, n - nr :], v[:, :, n - nr :]]
    for t, (q, k1, v1) in enumerate(d["steps"]):
        rec = [torch.cat([r, x.double()], dim=-2) for r, x in zip(rec, (k1, v1))]
        ks, vs = (torch.cat([s, h, r], dim=-2) for s, h, r in zip((out["sink_k"], out["sink_v"]), hat, rec))
        out["step%d" % t] = torch.stack([_softmax_rows(q[b], ks[b], vs[b]) for b in range(case["B"])])
    out["recent_k"], out["recent_v"] = rec
    return out


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_attention(case, seed)
    if kind == "compress":
        return _exact_compress(case, seed)
    if kind == "decompress":
        return _exact_decompress(case, seed)
    return _exact_layer(case, seed)
