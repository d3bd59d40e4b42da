"""What the speed of this framework is measured on.

Each case is one pass through public entry points: the device-pointer C ABI of
``include/tessera_gfx950.h``, bound by :mod:`tessera_amd.lane` and called on a PyTorch program's
tensors, or the device handles of :mod:`tessera_amd.resident`.  ``kind`` names the path:

``batched_gemm``  a stack of independent small products (``ops.batched_gemm``), f32 result
``gemm``          ``ops.gemm`` with the result in the operands' type
``gemm_act``      the fused bias + activation epilogue of a dense projection, f32 result
``attention``     flash attention forward: prefill, decode (few query rows), window, soft cap
``attn_train``    attention in a training step: forward with O and LSE saved, then dQ, dK, dV
``w8a8``          an int8 layer: per-row quantiser of the activation, then the scaled product
``fp8``           an fp8 layer: quantiser with a calibrated scale, then the scaled product
``moe``           the whole top-k SwiGLU expert layer: (router product,) routing, experts, combine
``attn_block``    a resident chain: fused QKV projection, attention on it in place, output projection

Sizes are those of the benchmark and the tests, or generic ones of the same order.
"""
from __future__ import annotations

import ctypes
import math

import torch

from tessera_amd import lane, resident

_DTYPE = {"bf16": torch.bfloat16, "f16": torch.float16}
_ACTIVATION = {"none": 0, "relu": 1, "gelu": 2, "silu": 3}
_F = ctypes.c_float


def listed():
    return [
        # The README's step of the reference: the smallest call, where the launch is what counts.
        {"name": "batched_small", "kind": "batched_gemm", "batch": 4, "m": 128, "n": 256, "k": 64, "dtype": "f16"},
        # A decode step's projection: a batch of 16 tokens against one big weight matrix.
        {"name": "gemm_decode", "kind": "gemm", "m": 16, "n": 8192, "k": 8192, "dtype": "bf16"},
        # An MLP up-projection over a prompt of an odd length, bias and GELU in the epilogue.
        {"name": "gemm_ragged_gelu", "kind": "gemm_act", "m": 1531, "n": 14336, "k": 4096, "dtype": "f16", "act": "gelu"},
        # The headline product: training and large prefill.
        {"name": "gemm_prefill", "kind": "gemm", "m": 8192, "n": 8192, "k": 8192, "dtype": "bf16"},
        # An attention block over two prompts of 500 tokens, as a Python chain on device handles.
        {"name": "attn_block_ragged", "kind": "attn_block", "batch": 2, "seq": 500, "hidden": 4096, "hq": 32, "hkv": 8,
         "d": 128, "dtype": "bf16"},
        # Causal grouped-query prefill over long prompts.
        {"name": "attn_prefill", "kind": "attention", "batch": 4, "hq": 32, "hkv": 8, "sq": 4096, "sk": 4096, "d": 128,
         "causal": True, "window": 0, "softcap": 0.0, "dtype": "bf16"},
        # One new token for each of 64 sequences against a cache of 2048 keys.
        {"name": "attn_decode", "kind": "attention", "batch": 64, "hq": 32, "hkv": 8, "sq": 1, "sk": 2048, "d": 128,
         "causal": False, "window": 0, "softcap": 0.0, "dtype": "bf16"},
        # Forward and backward of the same attention in a training step.
        {"name": "attn_train", "kind": "attn_train", "batch": 4, "hq": 32, "hkv": 8, "sq": 4096, "sk": 4096, "d": 128,
         "causal": True, "dtype": "bf16"},
        # Quantised serving: 16 tokens through an int8 layer (weight read once).
        {"name": "w8a8_decode", "kind": "w8a8", "m": 16, "n": 8192, "k": 8192},
        # Quantised prefill: 4096 tokens through an fp8 layer.
        {"name": "fp8_prefill", "kind": "fp8", "m": 4096, "n": 8192, "k": 8192, "format": "e4m3"},
        # Expert layer in decode: 64 tokens, every expert's weights are read for a handful of rows.
        {"name": "moe_decode", "kind": "moe", "tokens": 64, "hidden": 4096, "ffn": 1408, "experts": 64, "top_k": 8,
         "router": True},
        # Expert layer in prefill, the largest configuration of the benchmark; routing decided by the caller's logits.
        {"name": "moe_prefill", "kind": "moe", "tokens": 8192, "hidden": 4096, "ffn": 1408, "experts": 64, "top_k": 8,
         "router": False},
    ]


def _log(rng, low, high, multiple=1):
    """A whole number spread over the logarithm of [low, high], a multiple of ``multiple``."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(multiple, int(round(v / multiple)) * multiple)


def _width(rng, low, high):
    """A matrix width: mostly a multiple of 64, now and then any multiple of 8 or any number."""
    return _log(rng, low, high, rng.choice((64, 64, 64, 64, 8, 1)))


def draw(rng):
    kind = rng.choice(("batched_gemm", "gemm", "gemm", "gemm_act", "attn_block", "attention", "attention", "attn_train",
                       "w8a8", "fp8", "moe", "moe"))
    dtype = rng.choice(("bf16", "bf16", "f16"))
    most = 1.1e12                                     # multiply-adds are two: the headline product
    if kind == "batched_gemm":
        c = {"kind": kind, "batch": _log(rng, 2, 64), "m": _log(rng, 16, 1024), "n": _width(rng, 64, 1024),
             "k": _width(rng, 64, 1024), "dtype": dtype}
    elif kind in ("gemm", "gemm_act"):
        c = {"kind": kind, "m": _log(rng, 1, 8192), "n": _width(rng, 512, 16384), "k": _width(rng, 512, 14336),
             "dtype": dtype}
        if kind == "gemm_act":
            c["act"] = rng.choice(("none", "relu", "gelu", "silu"))
    elif kind == "attn_block":
        heads, group, d = rng.choice((8, 16, 32)), rng.choice((1, 4, 8)), rng.choice((64, 128))
        c = {"kind": kind, "batch": _log(rng, 1, 16), "seq": _log(rng, 8, 2048), "hidden": heads * d, "hq": heads,
             "hkv": heads // group, "d": d, "dtype": dtype}
    elif kind == "attention":
        heads, group, d = rng.choice((8, 16, 32)), rng.choice((1, 4, 8)), rng.choice((64, 64, 80, 128, 128, 128, 256))
        c = {"kind": kind, "batch": _log(rng, 1, 64), "hq": heads, "hkv": heads // group, "d": d, "dtype": dtype}
        if rng.random() < 0.5:                        # decode: one query row, or a few of a speculative step
            c.update(sq=rng.choice((1, 1, 1, 4)), sk=_log(rng, 64, 16384), causal=False, window=0, softcap=0.0)
            c["causal"] = c["sq"] > 1
        else:
            s = _log(rng, 64, 4096)
            c.update(sq=s, sk=s + rng.choice((0, 0, 0, _log(rng, 16, 1024))), causal=rng.random() < 0.8,
                     window=rng.choice((0, 0, 0, _log(rng, 32, 1024))), softcap=rng.choice((0.0, 0.0, 0.0, 30.0)))
    elif kind == "attn_train":
        heads, group, d = rng.choice((8, 16, 32)), rng.choice((1, 4, 8)), rng.choice((64, 128, 128))
        s = _log(rng, 128, 4096)
        c = {"kind": kind, "batch": _log(rng, 1, 16), "hq": heads, "hkv": heads // group, "sq": s, "sk": s, "d": d,
             "causal": rng.random() < 0.8, "dtype": dtype}
    elif kind == "w8a8":
        c = {"kind": kind, "m": _log(rng, 1, 4096), "n": _width(rng, 512, 14336), "k": _width(rng, 512, 14336)}
    elif kind == "fp8":
        c = {"kind": kind, "m": _log(rng, 1, 4096), "n": _width(rng, 512, 14336), "k": _width(rng, 512, 14336),
             "format": rng.choice(("e4m3", "e4m3", "e5m2"))}
    else:
        experts = rng.choice((8, 16, 32, 64))
        c = {"kind": kind, "tokens": _log(rng, 1, 4096), "hidden": _log(rng, 1024, 4096, 64),
             "ffn": _log(rng, 512, 4096, 64), "experts": experts, "top_k": rng.choice((1, 2, 4, 8)),
             "router": rng.random() < 0.5}
        while 6.0 * c["experts"] * c["hidden"] * c["ffn"] > 2.3e9:
            c["ffn"] = max(512, c["ffn"] // 128 * 64)
            if c["ffn"] == 512:
                c["experts"] = min(c["experts"], 32)
                break
    # the batch (or the rows) gives way where a draw would cost more than the largest listed case
    for size in ("batch", "m", "tokens"):
        while size in c and c[size] > 1 and (work(c)["flops"] > most or work(c)["bytes"] > 3e9):
            c[size] = c[size] // 2
    return c


def _randn(gen, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * scale).to(dtype)


def _weights(gen, experts, rows, cols):
    """Expert weights N(0, 0.02), drawn one expert at a time (the f32 draw is a temporary)."""
    w = torch.empty((experts, rows, cols), device="cuda", dtype=torch.bfloat16)
    for e in range(experts):
        w[e].copy_(torch.randn((rows, cols), generator=gen, device="cuda") * 0.02)
    return w


class _Exported:
    """A resident result seen by PyTorch without a copy (the tensor keeps the handle alive)."""

    def __init__(self, array):
        kind = {"bf16": "<i2", "f16": "<f2", "f32": "<f4"}[array.dtype]
        self.array = array
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": kind, "data": (array.ptr, False),
                                         "version": 2, "strides": None}


def _as_tensor(array):
    t = torch.as_tensor(_Exported(array), device="cuda")
    return t.view(torch.bfloat16) if array.dtype == "bf16" else t


def _resident(lib, t, dtype):
    """A device handle holding a copy of a tensor."""
    a = resident.DeviceArray(tuple(t.shape), dtype)
    lane.check(lib.tessera_gfx950_memcpy_d2d_dev(a.ptr, t.data_ptr(), a.nbytes // 16 * 16, None), "copy")
    torch.cuda.synchronize()
    return a


def prepare(case, seed):
    lib = lane.load()
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    s = {"case": case, "lib": lib, "stream": torch.cuda.current_stream().cuda_stream}
    new = lambda shape, dtype: torch.zeros(shape, device="cuda", dtype=dtype)  # noqa: E731
    if kind in ("batched_gemm", "gemm", "gemm_act"):
        dt, lead = _DTYPE[case["dtype"]], (case["batch"],) if kind == "batched_gemm" else ()
        m, n, k = case["m"], case["n"], case["k"]
        s["a"] = _randn(gen, lead + (m, k), dt, k ** -0.5)
        s["b"] = _randn(gen, lead + (k, n), dt, 1.0)
        s["out"] = new(lead + (m, n), dt if kind == "gemm" else torch.float32)
        name = {"batched_gemm": "batched_gemm_" + case["dtype"], "gemm": "gemm_%s_%s" % (case["dtype"], case["dtype"]),
                "gemm_act": "gemm_bias_act_" + case["dtype"]}[kind]
        s["fn"] = getattr(lib, "tessera_gfx950_%s_dev" % name)
        if kind == "gemm_act":
            s["bias"] = _randn(gen, (n,), torch.float32)
    elif kind in ("attention", "attn_train"):
        dt = _DTYPE[case["dtype"]]
        b, hq, hkv, sq, sk, d = (case[x] for x in ("batch", "hq", "hkv", "sq", "sk", "d"))
        s["q"] = _randn(gen, (b, hq, sq, d), dt)
        s["k"], s["v"] = _randn(gen, (b, hkv, sk, d), dt), _randn(gen, (b, hkv, sk, d), dt)
        s["o"], s["lse"] = new((b, hq, sq, d), dt if kind == "attention" else torch.float32), new((b, hq, sq), torch.float32)
        plain = kind == "attn_train" or not (case["window"] or case["softcap"])
        s["fn"] = getattr(lib, "tessera_gfx950_flash_attn_%s_%s_dev" % ("gqa" if plain else "ext", case["dtype"]))
        s["extra"] = () if plain else (case["window"], _F(case["softcap"]))
        if kind == "attn_train":
            s["do"] = _randn(gen, (b, hq, sq, d), dt)
            s["dq"], s["dk"], s["dv"] = (new(s[x].shape, torch.float32) for x in ("q", "k", "v"))
            s["bwd"] = getattr(lib, "tessera_gfx950_flash_attn_bwd_%s_dev" % case["dtype"])
    elif kind in ("w8a8", "fp8"):
        m, n, k = case["m"], case["n"], case["k"]
        s["x"] = _randn(gen, (m, k), torch.float32)
        w = _randn(gen, (k, n), torch.float32, k ** -0.5)
        s["xq"], s["wq"] = new((m, k), torch.int8 if kind == "w8a8" else torch.uint8), new((k, n), torch.int8)
        if kind == "w8a8":
            s["row_scale"], s["col_scale"] = new((m,), torch.float32), new((n,), torch.float32)
            s["out"] = new((m, n), torch.float32)
            lane.check(lib.tessera_gfx950_quantize_i8_f32_dev(w.data_ptr(), k, n, 0, s["wq"].data_ptr(),
                                                              s["col_scale"].data_ptr(), s["stream"]), "quantise")
        else:
            top = 448.0 if case["format"] == "e4m3" else 57344.0
            s["scale_x"] = 5.0 / top                  # a calibrated range: a few values beyond it are clipped
            s["scale_w"] = float(w.abs().max()) / top
            s["scale_out"] = new((1,), torch.float32)
            s["out"] = new((m, n), torch.bfloat16)
            s["quantise"] = getattr(lib, "tessera_gfx950_quantize_%s_f32_dev" % case["format"])
            s["fn"] = getattr(lib, "tessera_gfx950_gemm_%s_bf16_dev" % case["format"])
            lane.check(s["quantise"](w.data_ptr(), k * n, _F(s["scale_w"]), s["wq"].data_ptr(), s["scale_out"].data_ptr(),
                                     s["stream"]), "quantise")
        torch.cuda.synchronize()
    elif kind == "moe":
        t, h, f, e, k = (case[x] for x in ("tokens", "hidden", "ffn", "experts", "top_k"))
        s["x"] = _randn(gen, (t, h), torch.bfloat16)
        s["router"] = _randn(gen, (h, e), torch.bfloat16, h ** -0.5) if case["router"] else None
        s["logits"] = None if case["router"] else _randn(gen, (t, e), torch.float32)
        s["wg"], s["wu"], s["wd"] = _weights(gen, e, h, f), _weights(gen, e, h, f), _weights(gen, e, f, h)
        s["out"] = new((t, h), torch.float32)
        s["plan"] = [new((t * k,), torch.int32), new((t * k,), torch.int32), new((t * k,), torch.float32),
                     new((e,), torch.int32), new((e + 1,), torch.int32), new((1,), torch.int32)]
        need = ctypes.c_size_t(0)
        lane.check(lib.tessera_gfx950_moe_layer_workspace_bytes(t, h, f, h, e, k, ctypes.byref(need)), "workspace")
        s["workspace"] = torch.empty((need.value,), device="cuda", dtype=torch.uint8)
    else:
        dt, h, d = _DTYPE[case["dtype"]], case["hidden"], case["d"]
        width = (case["hq"] + 2 * case["hkv"]) * d
        s["x"] = _resident(lib, _randn(gen, (case["batch"] * case["seq"], h), dt), case["dtype"])
        s["wqkv"] = _resident(lib, _randn(gen, (h, width), dt, h ** -0.5), case["dtype"])
        s["wo"] = _resident(lib, _randn(gen, (case["hq"] * d, h), dt, (case["hq"] * d) ** -0.5), case["dtype"])
    return s


def run(s):
    c, lib, stream, kind = s["case"], s["lib"], s["stream"], s["case"]["kind"]
    if kind == "batched_gemm":
        lane.check(s["fn"](s["a"].data_ptr(), s["b"].data_ptr(), s["out"].data_ptr(), c["batch"], c["m"], c["n"], c["k"],
                           stream), kind)
        return s["out"]
    if kind == "gemm":
        lane.check(s["fn"](s["a"].data_ptr(), s["b"].data_ptr(), s["out"].data_ptr(), c["m"], c["n"], c["k"], stream), kind)
        return s["out"]
    if kind == "gemm_act":
        lane.check(s["fn"](s["a"].data_ptr(), s["b"].data_ptr(), s["bias"].data_ptr(), _ACTIVATION[c["act"]],
                           s["out"].data_ptr(), c["m"], c["n"], c["k"], stream), kind)
        return s["out"]
    if kind in ("attention", "attn_train"):
        dims = (c["batch"], c["hq"], c["hkv"], c["sq"], c["sk"], c["d"], _F(c["d"] ** -0.5), int(c["causal"]))
        q, k, v, o, lse = (s[x].data_ptr() for x in ("q", "k", "v", "o", "lse"))
        if kind == "attention":
            lane.check(s["fn"](q, k, v, o, lse, *dims, *s["extra"], 1, stream), kind)
            return s["o"], s["lse"]
        lane.check(s["fn"](q, k, v, o, lse, *dims, 0, stream), kind)
        lane.check(s["bwd"](s["do"].data_ptr(), q, k, v, o, lse, s["dq"].data_ptr(), s["dk"].data_ptr(),
                            s["dv"].data_ptr(), *dims, stream), kind)
        return s["o"], s["dq"], s["dk"], s["dv"]
    if kind == "w8a8":
        m, n, k = c["m"], c["n"], c["k"]
        xq, rs = s["xq"].data_ptr(), s["row_scale"].data_ptr()
        lane.check(lib.tessera_gfx950_quantize_i8_f32_dev(s["x"].data_ptr(), m, k, 1, xq, rs, stream), "quantise")
        lane.check(lib.tessera_gfx950_gemm_w8a8_f32_dev(xq, s["wq"].data_ptr(), rs, s["col_scale"].data_ptr(),
                                                        s["out"].data_ptr(), None, m, n, k, stream), kind)
        return s["out"], s["xq"], s["row_scale"]
    if kind == "fp8":
        m, n, k = c["m"], c["n"], c["k"]
        xq = s["xq"].data_ptr()
        lane.check(s["quantise"](s["x"].data_ptr(), m * k, _F(s["scale_x"]), xq, s["scale_out"].data_ptr(), stream), "quantise")
        lane.check(s["fn"](xq, s["wq"].data_ptr(), _F(s["scale_x"]), _F(s["scale_w"]), s["out"].data_ptr(), m, n, k, stream),
                   kind)
        return s["out"], s["xq"]
    if kind == "moe":
        t, h, f, e, k = (c[x] for x in ("tokens", "hidden", "ffn", "experts", "top_k"))
        lane.check(lib.tessera_gfx950_moe_layer_bf16_dev(
            s["x"].data_ptr(), s["router"].data_ptr() if c["router"] else None,
            None if c["router"] else s["logits"].data_ptr(), s["wg"].data_ptr(), s["wu"].data_ptr(), s["wd"].data_ptr(),
            s["out"].data_ptr(), s["workspace"].data_ptr(), s["workspace"].numel(), t, h, f, h, e, k, 1, 0,
            *(p.data_ptr() for p in s["plan"]), stream), kind)
        # with the logits given the plan is exact; a router product in another order may break a tie the other way
        return s["out"] if c["router"] else (s["out"], *s["plan"])
    qkv = resident.gemm(s["x"], s["wqkv"]).reshape(c["batch"], c["seq"], (c["hq"] + 2 * c["hkv"]) * c["d"])
    o = resident.flash_attn_fused_qkv(qkv, c["hq"], c["hkv"], causal=True)
    y = resident.gemm(o.reshape(c["batch"] * c["seq"], c["hq"] * c["d"]), s["wo"])
    return _as_tensor(y)


def _pairs(sq, sk, causal, window):
    """Visible (query, key) pairs of one head."""
    if not causal and not window:
        return float(sq) * sk
    total, shift = 0, max(sk - sq, 0)
    for i in range(sq):
        at = i + shift
        if causal:
            low, high = (at - window + 1 if window else 0), at
        else:
            low, high = at - window // 2, at + window // 2
        total += max(0, min(high, sk - 1) - max(low, 0) + 1)
    return float(total)


def work(case):
    kind = case["kind"]
    if kind in ("batched_gemm", "gemm", "gemm_act"):
        batch, m, n, k = case.get("batch", 1), case["m"], case["n"], case["k"]
        out = (2 if kind == "gemm" else 4) * m * n + (4 * n if kind == "gemm_act" else 0)
        return {"bytes": batch * (2 * (m * k + k * n) + out), "flops": 2.0 * batch * m * n * k}
    if kind in ("attention", "attn_train"):
        b, hq, hkv, sq, sk, d = (case[x] for x in ("batch", "hq", "hkv", "sq", "sk", "d"))
        q, kv = b * hq * sq * d, b * hkv * sk * d
        flops = 4.0 * b * hq * d * _pairs(sq, sk, case["causal"], case.get("window", 0))
        if kind == "attention":
            return {"bytes": 2 * q + 4 * kv + 2 * q + 4 * b * hq * sq, "flops": flops}
        # the backward's five products against the forward's two
        return {"bytes": 4 * q + 4 * kv + 4 * q + 4 * q + 8 * kv, "flops": 3.5 * flops}
    if kind in ("w8a8", "fp8"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * m * k + m * k + k * n + (4 if kind == "w8a8" else 2) * m * n, "flops": 2.0 * m * n * k}
    if kind == "moe":
        t, h, f, e, k = (case[x] for x in ("tokens", "hidden", "ffn", "experts", "top_k"))
        touched = e * (1.0 - (1.0 - min(1.0, k / e)) ** t)          # experts that some token is expected to choose
        return {"bytes": 6.0 * touched * h * f + 2 * t * h + 4 * t * h + (2 * h * e if case["router"] else 4 * t * e),
                "flops": 6.0 * t * k * h * f + (2.0 * t * h * e if case["router"] else 0)}
    t, h, d = case["batch"] * case["seq"], case["hidden"], case["d"]
    width = (case["hq"] + 2 * case["hkv"]) * d
    flops = 2.0 * t * h * (width + case["hq"] * d)
    flops += 4.0 * case["batch"] * case["hq"] * d * _pairs(case["seq"], case["seq"], True, 0)
    return {"bytes": 2 * (2 * t * h + h * width + h * case["hq"] * d), "flops": flops}


def tolerance(case):
    """About four times the relative error of the path against the same arithmetic in 64 bits (in brackets: measured)."""
    kind, f16 = case["kind"], case.get("dtype") == "f16"
    if kind in ("batched_gemm", "gemm_act"):
        return {"rel": 2e-6}                          # f32 results of f32 sums (6e-8 at K = 64, 2.8e-7 at K = 4096)
    if kind == "w8a8":
        return {"rel": 2e-7}                          # exact sums, codes and scales, two f32 multiplies (3.6e-8)
    if kind in ("gemm", "fp8", "attn_train"):
        return {"rel": 9e-4 if f16 else 7e-3}         # one rounding to 16 bits (f16 2.1e-4, bf16 1.7e-3)
    if kind == "attention":
        return {"rel": 1e-3 if f16 else 8e-3}         # probabilities and result rounded (f16 2.5e-4, bf16 2.1e-3)
    return {"rel": 2e-3 if f16 else 1.5e-2}           # three or four roundings in a chain (bf16 3.5e-3, 3.7e-3)
