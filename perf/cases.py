"""The work that programs have this package do, as cases that can be timed and compared.

A program built on the package runs a decoder: prompts go through the dense or the packed attention, tokens through the
decode attention over a KV cache (16-bit or Q8_0 blocks), and around both stand the normalisation, the projections and the
rotary embedding that appends to the cache.  Every case calls `minfer.kernels.KernelBackend("torch_ext")` the way such a
program does: outputs and caches are the caller's, activations are [B, L, heads * head_dim] and reach attention as
[B, heads, L, head_dim] views.  The number of tokens, of cached rows and of rows of an activation is whatever the prompts
and the batch happen to be; head counts, hidden sizes and weights are a model's.
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.abspath("minfer-python_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from minfer.const import GGML_QUANT_SIZES, GGMLQuantizationType  # noqa: E402
from minfer.kernels import KernelBackend  # noqa: E402

_KERNELS = KernelBackend("torch_ext")
_F16 = (int(GGMLQuantizationType.F16), *GGML_QUANT_SIZES[GGMLQuantizationType.F16])
_BF16 = (int(GGMLQuantizationType.BF16), *GGML_QUANT_SIZES[GGMLQuantizationType.BF16])
_Q8 = (int(GGMLQuantizationType.Q8_0), *GGML_QUANT_SIZES[GGMLQuantizationType.Q8_0])
_DEV = "cuda"
_EPS = 1e-6
_BASE = 5e5       # rotary frequency base
_NEOX = 1

# (query heads, KV heads) of the models' layers: grouped 4:1 in small and middle size, 1:1, 3:1, 6:1, 8:1
_HEADS = ((8, 2), (16, 16), (24, 8), (32, 8), (48, 8), (64, 8))
# (out, in) of projections: fused and single attention projections, feed-forward up, gate + up and down, narrow models, an output head
_WEIGHTS = ((6144, 4096), (4096, 4096), (14336, 4096), (28672, 4096), (4096, 14336), (8192, 8192), (2048, 8192), (1536, 8960), (128256, 4096))


def listed():
    return [
        # a short prompt on a small model (the repository's smallest configuration); the smallest call, latency only
        {"name": "prefill_short", "kind": "prefill", "B": 1, "Hq": 8, "Hkv": 2, "L": 256, "D": 64, "dtype": "f16", "window": 0},
        # a few prompts of no round length under a sliding window, as the reference's own test has it
        {"name": "prefill_window_odd", "kind": "prefill", "B": 4, "Hq": 32, "Hkv": 8, "L": 1003, "D": 128, "dtype": "bf16", "window": 256},
        # the headline: one 4096-token prompt at the 8B shape
        {"name": "prefill_4096", "kind": "prefill", "B": 1, "Hq": 32, "Hkv": 8, "L": 4096, "D": 128, "dtype": "f16", "window": 0},
        # a whole long document at once; the largest case
        {"name": "prefill_32768", "kind": "prefill", "B": 1, "Hq": 32, "Hkv": 8, "L": 32768, "D": 128, "dtype": "bf16", "window": 0},
        # prompts of a serving batch packed without padding, at the 70B head shape
        {"name": "packed_ragged", "kind": "packed", "n": 16, "lo": 128, "hi": 2048, "lens": 0, "Hq": 64, "Hkv": 8, "D": 128, "dtype": "f16"},
        # one decode step's attention of a full serving batch
        {"name": "decode_batch", "kind": "decode", "B": 64, "Hq": 32, "Hkv": 8, "D": 128, "lo": 512, "hi": 8192, "lens": 0, "dtype": "f16", "cache": "f16"},
        # the same for a few short conversations over a quantised cache
        {"name": "decode_q8_few", "kind": "decode", "B": 3, "Hq": 32, "Hkv": 8, "D": 128, "lo": 200, "hi": 3000, "lens": 1, "dtype": "f16", "cache": "q8_0"},
        # a whole attention block of one decode step for a single user: norm, QKV, rotary + append, attention, output + residual
        {"name": "step_single", "kind": "block", "B": 1, "L": 1, "past": 1500, "Hq": 32, "Hkv": 8, "D": 128, "dtype": "bf16", "cache": "bf16", "norm": False},
        # the same for a serving batch over a quantised cache
        {"name": "step_batch_q8", "kind": "block", "B": 40, "L": 1, "past": 1100, "Hq": 32, "Hkv": 8, "D": 128, "dtype": "f16", "cache": "q8_0", "norm": False},
        # the same block over a prompt of no round length, with the per-head normalisation of q and k
        {"name": "prompt_block", "kind": "block", "B": 1, "L": 1777, "past": 0, "Hq": 32, "Hkv": 8, "D": 128, "dtype": "f16", "cache": "f16", "norm": True},
        # a feed-forward projection of a decode batch against a quantised weight
        {"name": "project_q8_16", "kind": "project", "M": 16, "N": 14336, "K": 4096, "weight": "q8_0", "dtype": "f16", "residual": False},
        # a feed-forward projection of a prefill chunk
        {"name": "project_chunk", "kind": "project", "M": 600, "N": 14336, "K": 4096, "weight": "nk", "dtype": "bf16", "residual": False},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("prefill", "prefill", "prefill", "packed", "decode", "decode", "block", "block", "block", "project", "project", "project"))
    Hq, Hkv = rng.choice(_HEADS)
    dtype = rng.choice(("f16", "bf16"))
    D = rng.choice((64, 128, 128))
    if kind == "prefill":
        L = _log_int(rng, 24, 16384)
        B = _log_int(rng, 1, max(1, min(16, 16384 // L)))
        return {"kind": kind, "B": B, "Hq": Hq, "Hkv": Hkv, "L": L, "D": D, "dtype": dtype, "window": rng.choice((0, 0, 0, 256))}
    if kind == "packed":
        hi = _log_int(rng, 64, 4096)
        return {"kind": kind, "n": _log_int(rng, 2, min(64, max(2, 65536 // hi))), "lo": max(1, hi // 16), "hi": hi, "lens": rng.randrange(1 << 20),
                "Hq": Hq, "Hkv": Hkv, "D": D, "dtype": dtype}
    if kind == "decode":
        B = _log_int(rng, 1, 64)
        hi = _log_int(rng, 64, min(65536, 524288 // B))
        cache = rng.choice((dtype, dtype, "q8_0"))
        return {"kind": kind, "B": B, "Hq": Hq, "Hkv": Hkv, "D": D, "lo": max(1, hi // 16), "hi": hi, "lens": rng.randrange(1 << 20),
                "dtype": "f16" if cache == "q8_0" else dtype, "cache": cache}
    if kind == "block":
        cache = rng.choice((dtype, dtype, "q8_0"))
        dtype = "f16" if cache == "q8_0" else dtype
        norm = rng.choice((False, True))
        if rng.random() < 0.5:   # a decode step
            B = _log_int(rng, 1, 64)
            return {"kind": kind, "B": B, "L": 1, "past": _log_int(rng, 16, min(32768, 262144 // B)), "Hq": Hq, "Hkv": Hkv, "D": 128,
                    "dtype": dtype, "cache": cache, "norm": norm}
        return {"kind": kind, "B": 1, "L": _log_int(rng, 16, 8192), "past": 0, "Hq": Hq, "Hkv": Hkv, "D": 128, "dtype": dtype, "cache": cache, "norm": norm}
    if rng.random() < 0.5:
        N, K = rng.choice(_WEIGHTS)
    else:   # any model's sizes
        N, K = 8 * _log_int(rng, 64, 4096), 64 * _log_int(rng, 16, 256)
    weight = rng.choice(("nk", "nk", "kn", "q8_0"))
    M = _log_int(rng, 1, 64 if N > 100000 else 8192)
    return {"kind": kind, "M": M, "N": N, "K": K, "weight": weight, "dtype": "f16" if weight == "q8_0" else dtype, "residual": rng.choice((False, True))}


def _torch_dtype(name):
    return torch.bfloat16 if name == "bf16" else torch.float16


def _qt(name):
    return {"f16": _F16, "bf16": _BF16, "q8_0": _Q8}[name]


def _lens(case, n):
    r = random.Random(case["lens"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(n)]


class _Draw:
    """Tensors of normally distributed values on the GPU, one after the other from one seed."""

    def __init__(self, seed, dtype):
        self.gen = torch.Generator(device=_DEV).manual_seed(seed)
        self.dtype = dtype

    def __call__(self, *shape, scale=1.0):
        t = torch.randn(*shape, generator=self.gen, device=_DEV, dtype=self.dtype)
        return t.mul_(scale) if scale != 1.0 else t


def _blocks(x):
    """Rows of x as Q8_0 blocks, quantised by the package."""
    y = torch.empty(*x.shape[:-1], x.shape[-1] // 32 * 34, dtype=torch.uint8, device=x.device)
    _KERNELS._quant(*_Q8, x.reshape(-1, x.shape[-1]), y.view(-1, y.shape[-1]))
    return y


def _heads(x, H, D):
    """[B, L, H * D] as the [B, H, L, D] view that attention takes."""
    return x.view(x.shape[0], x.shape[1], H, D).transpose(1, 2)


def _mask(B, L, window):
    i = torch.arange(L, device=_DEV, dtype=torch.int32)
    m = i[None, :] <= i[:, None]
    if window:
        m &= i[None, :] > i[:, None] - window
    return m[None, None].expand(B, 1, L, L).contiguous()


def prepare(case, seed):
    kind, dtype = case["kind"], _torch_dtype(case["dtype"])
    rnd = _Draw(seed, dtype)
    s = {"case": case}
    if kind == "project":
        M, N, K = case["M"], case["N"], case["K"]
        s["x"] = rnd(1, M, K)
        w = rnd(*((K, N) if case["weight"] == "kn" else (N, K)), scale=K ** -0.5)
        s["w"] = _blocks(w) if case["weight"] == "q8_0" else w
        s["c"], s["out"] = rnd(1, M, N), torch.empty(1, M, N, dtype=dtype, device=_DEV)
        return s
    Hq, Hkv, D = case["Hq"], case["Hkv"], case["D"]
    if kind == "prefill":
        B, L = case["B"], case["L"]
        s["q"] = _heads(rnd(B, L, Hq * D, scale=0.5), Hq, D)
        s["k"], s["v"] = (_heads(rnd(B, L, Hkv * D, scale=0.5), Hkv, D) for _ in range(2))
        s["mask"] = _mask(B, L, case["window"])
        s["y"] = torch.empty(B, L, Hq * D, dtype=dtype, device=_DEV)
        s["out"] = _heads(s["y"], Hq, D)
    elif kind == "packed":
        lens = _lens(case, case["n"])
        T = sum(lens)
        s["q"] = _heads(rnd(1, T, Hq * D), Hq, D)
        s["k"], s["v"] = (_heads(rnd(1, T, Hkv * D), Hkv, D) for _ in range(2))
        s["cu"] = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device=_DEV)
        s["longest"] = max(lens)
        s["y"] = torch.empty(1, T, Hq * D, dtype=dtype, device=_DEV)
        s["out"] = _heads(s["y"], Hq, D)
    elif kind == "decode":
        B = case["B"]
        s["q"] = _heads(rnd(B, 1, Hq * D), Hq, D)
        s["kc"], s["vc"] = rnd(B, Hkv, case["hi"], D), rnd(B, Hkv, case["hi"], D)
        if case["cache"] == "q8_0":
            s["kc"], s["vc"] = _blocks(s["kc"]), _blocks(s["vc"])
        s["ctx"] = torch.tensor(_lens(case, B), dtype=torch.int32, device=_DEV)
        s["y"] = torch.empty(B, 1, Hq * D, dtype=dtype, device=_DEV)
        s["out"] = _heads(s["y"], Hq, D)
    else:   # block
        B, L, past, hidden = case["B"], case["L"], case["past"], Hq * D
        s["x"] = rnd(B, L, hidden)
        s["w_in"] = rnd(hidden, scale=0.1).add_(1.0)
        s["wq"], s["wk"], s["wv"] = (rnd(n * D, hidden, scale=hidden ** -0.5) for n in (Hq, Hkv, Hkv))
        s["wo"] = rnd(hidden, hidden, scale=hidden ** -0.5)
        s["wq_norm"], s["wk_norm"] = (rnd(D, scale=0.1).add_(1.0) for _ in range(2))
        s["kc"], s["vc"] = rnd(B, Hkv, past + L, D), rnd(B, Hkv, past + L, D)
        if case["cache"] == "q8_0":
            s["kc"], s["vc"] = _blocks(s["kc"]), _blocks(s["vc"])
        s["pos"] = torch.full((B,), past, dtype=torch.int32, device=_DEV)
        s["ctx"] = torch.full((B,), past + 1, dtype=torch.int32, device=_DEV)
        if L > 1:
            s["mask"] = _mask(B, L, 0)
        for name, width in (("h", hidden), ("q", hidden), ("k", Hkv * D), ("v", Hkv * D), ("a", hidden), ("y", hidden)):
            s[name] = torch.empty(B, L, width, dtype=dtype, device=_DEV)
    return s


def _block(s, case):
    B, L, Hq, Hkv, D = (case[n] for n in ("B", "L", "Hq", "Hkv", "D"))
    kt, act = _qt(case["cache"]), _qt(case["dtype"])
    _KERNELS.rmsnorm(_EPS, s["x"], s["w_in"], s["h"])
    _KERNELS.qkv(*(t for three in zip(act, act, act) for t in three), s["h"], s["wq"], s["wk"], s["wv"], s["q"], s["k"], s["v"])
    q, k, v = s["q"].view(B, L, Hq, D), s["k"].view(B, L, Hkv, D), s["v"].view(B, L, Hkv, D)
    if case["norm"]:
        _KERNELS.rope_kv_append_norm(_NEOX, D, _BASE, _EPS, q, k, v, s["wq_norm"], s["wk_norm"], s["pos"], s["kc"], s["vc"])
    else:
        _KERNELS.rope_kv_append(_NEOX, D, _BASE, q, k, v, s["pos"], s["kc"], s["vc"])
    if L == 1:
        _KERNELS.flash_attn_decode(*kt, q.transpose(1, 2), s["kc"], s["vc"], s["ctx"], _heads(s["a"], Hq, D))
    else:
        _KERNELS.flash_attn(*kt, q.transpose(1, 2), s["kc"], s["vc"], s["mask"], _heads(s["a"], Hq, D))
    _KERNELS.gemm(*act, 1.0, 1.0, s["a"], s["wo"], s["x"], s["y"])
    return {"y": s["y"], "kc": s["kc"], "vc": s["vc"]}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "project":
        qt = _Q8 if case["weight"] == "q8_0" else _qt(case["dtype"])
        _KERNELS.gemm(*qt, 1.0, 1.0 if case["residual"] else 0.0, s["x"], s["w"], s["c"], s["out"])
        return s["out"]
    if kind == "prefill":
        _KERNELS.flash_attn(*_qt(case["dtype"]), s["q"], s["k"], s["v"], s["mask"], s["out"])
    elif kind == "packed":
        _KERNELS.flash_attn_varlen(*_qt(case["dtype"]), s["q"], s["k"], s["v"], s["cu"], s["longest"], s["out"])
    elif kind == "decode":
        _KERNELS.flash_attn_decode(*_qt(case["cache"]), s["q"], s["kc"], s["vc"], s["ctx"], s["out"])
    else:
        return _block(s, case)
    return s["y"]


def _pairs(L, window):
    """(query, key) pairs that a causal mask of L tokens lets through."""
    w = min(window or L, L)
    return w * (w + 1) // 2 + (L - w) * w


def work(case):
    kind = case["kind"]
    if kind == "project":
        M, N, K = case["M"], case["N"], case["K"]
        weight = N * K // 32 * 34 if case["weight"] == "q8_0" else 2 * N * K
        return {"bytes": weight + 2 * M * K + 2 * M * N * (2 if case["residual"] else 1), "flops": 2 * M * N * K}
    Hq, Hkv, D = case["Hq"], case["Hkv"], case["D"]
    row = D // 32 * 34 if case.get("cache") == "q8_0" else 2 * D   # bytes of one cached row of one head
    if kind == "prefill":
        B, L = case["B"], case["L"]
        return {"bytes": B * (L * (2 * Hq + 2 * Hkv) * D * 2 + L * L), "flops": 4 * D * Hq * B * _pairs(L, case["window"])}
    if kind == "packed":
        lens = _lens(case, case["n"])
        return {"bytes": sum(lens) * (2 * Hq + 2 * Hkv) * D * 2, "flops": 4 * D * Hq * sum(_pairs(n, 0) for n in lens)}
    if kind == "decode":
        rows = sum(_lens(case, case["B"]))
        return {"bytes": rows * Hkv * 2 * row + case["B"] * Hq * D * 4, "flops": 4 * D * Hq * rows}
    B, L, past, hidden = case["B"], case["L"], case["past"], Hq * D
    weights = hidden * (2 * hidden + 2 * Hkv * D)
    pairs = B * (_pairs(L, 0) + past)
    return {"bytes": 2 * weights + 2 * 2 * B * L * hidden + B * (past + L) * Hkv * 2 * row + (B * L * L if L > 1 else 0),
            "flops": 2 * B * L * weights + 4 * D * Hq * pairs}


def tolerance(case):
    # one rounding to the activation type (2^-11, 2^-8) of the result, of the attention weights before it and, in a block,
    # of every intermediate tensor; a Q8_0 cache keeps its bytes except where a value that it quantises was rounded the other way
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3, "differ": 0.01 if case.get("cache") == "q8_0" else 0.0}
