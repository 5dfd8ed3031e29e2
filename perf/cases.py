"""The work a user of this framework has it do, as measurable cases.

The framework is the quantisation path of an inference program: the element-wise operators that turn activations and
weights into and out of their quantised forms, and the quantised matmuls of a transformer's linear layers - int8 x int8
with dynamic activation scales, half x int4, half x int8, block-scaled (MX) fp8 / fp4, and the grouped matmul of a
mixture of experts.  Every matmul is met in two ways: prefill (hundreds to thousands of rows: arithmetic) and decode
(one to a few dozen rows: the weights' trip from memory, latency and launches).  Sizes are those of this repository's
benchmark and tests, or generic.

A case is a dict of plain values; `kind` says which path it takes:

  quant      activations to int8 / fp8 / fp4 codes      (ascend_quant, ascend_quant_policy, dynamic_quant_per_token)
  dequant    int32 accumulators to bf16 / fp32          (ascend_dequant)
  antiquant  int8 / int4 / fp8 / fp4 weights to half    (ascend_antiquant, ascend_antiquant_policy)
  linear     W8A8 linear: per-token quantisation of x, int8 matmul, de-quantising epilogue
  w4a16      half x int4 (per-group scale and offset)
  w8a16      half x int8 (per-channel scale and offset)
  moe        grouped W8A8 matmul, experts of uneven size
  mx         block-scaled matmul, fp8 / fp4 operands with one e8m0 scale per 32 k
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "asc-devkit_amd"))
from ascq import _abi as abi  # noqa: E402
from ascq import ops  # noqa: E402

DEV = "cuda"
FLOATS = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
SIZE = {"f16": 2, "bf16": 2, "f32": 4, "i8": 1, "e4m3": 1, "e5m2": 1, "i4": 0.5, "e2m1": 0.5, "e1m2": 0.5}
MX_FORMAT = {"e4m3": abi.QDST_FP8_E4M3FN, "e5m2": abi.QDST_FP8_E5M2, "e2m1": abi.QDST_FP4_E2M1, "e1m2": abi.QDST_FP4_E1M2}
ACT = {"none": abi.MM_ACT_NONE, "gelu": abi.MM_ACT_FASTER_GELU, "swiglu": abi.MM_ACT_SWIGLU}


def listed():
    return [
        # a layer's activations quantised with calibrated per-channel scales (static quantisation of a prefill batch)
        {"name": "quant_channel_8192x4096", "kind": "quant", "policy": "channel", "m": 8192, "n": 4096, "src": "f16", "dst": "i8"},
        # accumulators of an int8 matmul that ran without its epilogue, brought back to bf16
        {"name": "dequant_8192x4096", "kind": "dequant", "policy": "channel", "m": 8192, "n": 4096, "dst": "bf16"},
        # int4 weights of a feed-forward projection expanded to half once per use (per-group parameters)
        {"name": "antiquant_i4_group_4096x11008", "kind": "antiquant", "src": "i4", "m": 4096, "n": 11008, "groups": 32,
         "transposed": False, "offset": True, "dst": "f16"},
        # decode, one sequence: the smallest call, on weights packed when the model was loaded
        {"name": "linear_decode_m1", "kind": "linear", "m": 1, "k": 4096, "n": 11008, "weights": "packed", "act": "none",
         "bias": "none", "x": "bf16", "out": "bf16"},
        # a vision tower's second projection: token count, k and n off every tile size
        {"name": "linear_ragged_m729_k4304", "kind": "linear", "m": 729, "k": 4304, "n": 1152, "weights": "kn", "act": "none",
         "bias": "f32", "x": "f16", "out": "f16"},
        # prefill of 2048 tokens: the benchmark's headline
        {"name": "linear_prefill_m2048", "kind": "linear", "m": 2048, "k": 4096, "n": 11008, "weights": "kn", "act": "none",
         "bias": "none", "x": "bf16", "out": "bf16"},
        # decode with int4 weights, one sequence: the benchmark's second headline
        {"name": "w4a16_decode_m1", "kind": "w4a16", "m": 1, "k": 8192, "n": 28672, "weights": "packed", "mode": "group_sum",
         "group": 128, "offset": True},
        # prefill of a short prompt on the same int4 weights
        {"name": "w4a16_prefill_m512", "kind": "w4a16", "m": 512, "k": 8192, "n": 28672, "weights": "packed", "mode": "per_weight",
         "group": 128, "offset": True},
        # prefill with int8 weights and half activations
        {"name": "w8a16_prefill_m2048", "kind": "w8a16", "m": 2048, "k": 8192, "n": 28672, "weights": "nk", "mode": "per_weight",
         "per_tensor": False, "offset": True, "out": "f16"},
        # up projection of a mixture of experts, tokens routed at random
        {"name": "moe_prefill_8x4096", "kind": "moe", "groups": 8, "tokens": 4096, "k": 4096, "n": 14336, "weights": "nd", "act": "none",
         "bias": "bf16", "out": "bf16", "skew": 0.0},
        # decode batch of 16 sequences on fp4 weights
        {"name": "mx_decode_m16", "kind": "mx", "m": 16, "n": 8192, "k": 8192, "a": "e2m1", "b": "e2m1", "out": "bf16", "bias": False},
        # the block-scaled matmul at the size of the reference's own example, in its format
        {"name": "mx_prefill_8192_e1m2", "kind": "mx", "m": 8192, "n": 8192, "k": 8192, "a": "e1m2", "b": "e1m2", "out": "bf16",
         "bias": False},
    ]


# ---------------------------------------------------------------------------------------------------------- draws
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, q):
    """a multiple of q between lo and hi, spread over the logarithm"""
    return max(q, _log(rng, lo, hi) // q * q)


def draw(rng):
    kind = rng.choice(["quant", "dequant", "antiquant", "linear", "linear", "w4a16", "w8a16", "moe", "mx", "mx"])
    return {"kind": kind, **globals()["_draw_" + kind](rng)}


def _plane(rng, q, most):
    """rows x columns of an activation or weight matrix of up to `most` elements"""
    n = _mult(rng, 512, 16384, q)
    return _log(rng, 16, max(16, min(8192, most // n))), n


def _draw_quant(rng):
    policy = rng.choice(["channel", "tensor", "token", "group", "dynamic"])
    # parameter rows along the channels may have any width; the others keep the operator's 32-byte rows
    m, n = _plane(rng, rng.choice([1, 8, 128]) if policy in ("channel", "dynamic") else rng.choice([32, 128]), 32 << 20)
    src = rng.choice(["f16", "bf16", "f32"])
    dst = "i8"
    if policy in ("token", "group"):
        dst = rng.choice(["i8", "e4m3", "e5m2"] + (["e2m1"] if policy == "group" and src != "f32" else []))
    return {"policy": policy, "m": m, "n": n, "src": src, "dst": dst}


def _draw_dequant(rng):
    m, n = _plane(rng, rng.choice([8, 128]), 32 << 20)
    return {"policy": rng.choice(["channel", "tensor", "token", "group"]), "m": m, "n": n, "dst": rng.choice(["bf16", "f32"])}


def _draw_antiquant(rng):
    src = rng.choice(["i8", "i4", "e4m3", "e2m1"])
    k = _mult(rng, 512, 8192, 128)
    transposed = src in ("i8", "i4") and rng.random() < 0.5
    # rows of any width where the operator takes them (int8, not transposed)
    n = _mult(rng, 512, 14336, rng.choice([1, 16, 128]) if src == "i8" and not transposed else 64)
    if transposed or src not in ("i8", "i4"):
        m = n
        n = k
    else:
        m = k
    return {"src": src, "m": m, "n": n, "groups": rng.choice([1, k // 128]), "transposed": transposed,
            "offset": src != "e2m1" and rng.random() < 0.5, "dst": rng.choice(["f16", "bf16"])}


def _draw_linear(rng):
    act = rng.choice(["none", "none", "none", "gelu", "swiglu"])
    weights = rng.choice(["kn", "nk", "packed"])
    k = _mult(rng, 512, 11008, rng.choice([128, 128, 64] if weights == "packed" else [128, 128, 16]))
    n = _mult(rng, 256, 22016, rng.choice([128, 16, 8]))
    m = _log(rng, 1, min(4096, 2 ** 37 // (k * n)))
    if rng.random() < 0.15:
        # a vocabulary with added tokens: an odd number of columns, a few rows
        act, n, m = "none", _mult(rng, 2048, 32768, 16) + 2 * rng.randrange(8) + 1, min(m, _log(rng, 1, 32))
    return {"m": m, "k": k, "n": n, "weights": weights, "act": act, "bias": rng.choice(["none", "f32", "bf16"]),
            "x": rng.choice(["bf16", "f16"]), "out": rng.choice(["bf16", "f16"])}


def _draw_w4a16(rng):
    k, n = _mult(rng, 1024, 14336, 128), _mult(rng, 1024, 28672, rng.choice([32, 128]))
    weights = rng.choice(["packed", "packed", "nd"])
    return {"m": _log(rng, 1, min(2048, 2 ** 37 // (k * n))), "k": k, "n": n, "weights": weights,
            "mode": rng.choice(["per_weight", "group_sum"]) if weights == "packed" else "per_weight",
            "group": rng.choice([128, 128, 64]), "offset": rng.random() < 0.5}


def _draw_w8a16(rng):
    k, n = _mult(rng, 1024, 14336, 128), _mult(rng, 1024, 28672, rng.choice([16, 128]))
    return {"m": _log(rng, 1, min(4096, 2 ** 38 // (k * n))), "k": k, "n": n, "weights": rng.choice(["nk", "nk", "kn"]),
            "mode": rng.choice(["per_weight", "channel_sum"]), "per_tensor": rng.random() < 0.25, "offset": rng.random() < 0.5,
            "out": rng.choice(["f16", "f32"])}


def _draw_moe(rng):
    groups = rng.choice([4, 8, 16, 32])
    k, n = _mult(rng, 1024, 4096, 128), _mult(rng, 1024, 14336, rng.choice([32, 128]))
    while groups * k * n > 480 << 20:
        groups //= 2
    act = rng.choice(["none", "gelu", "swiglu"])
    return {"groups": groups, "tokens": _log(rng, 8, 8192 if k * n <= 24 << 20 else 4096), "k": k, "n": n,
            "weights": rng.choice(["nd", "nd", "nz"]), "act": act, "bias": rng.choice(["none", "bf16"]),
            "out": rng.choice(["bf16", "f16"]), "skew": rng.choice([0.0, 1.0])}


def _draw_mx(rng):
    a, b = rng.choice([("e4m3", "e4m3"), ("e2m1", "e2m1"), ("e1m2", "e1m2"), ("e5m2", "e4m3"), ("e4m3", "e2m1")])
    # half of the draws decode, half prefill
    decode = rng.random() < 0.5
    k, n = _mult(rng, 1024, 14336, 128 if decode else 256), _mult(rng, 1024, 14336, rng.choice([16, 128]))
    m = _log(rng, 1, 48) if decode else _log(rng, 64, min(8192, 2 ** 39 // (k * n)))
    return {"m": m, "n": n, "k": k, "a": a, "b": b, "out": rng.choice(["bf16", "f16", "f32"]), "bias": rng.random() < 0.25}


# ------------------------------------------------------------------------------------------------------ preparation
class _Source:
    """seeded inputs on the GPU"""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, std=1.0):
        return torch.empty(shape, dtype=torch.float32, device=DEV).normal_(0.0, std, generator=self.g).to(dtype)

    def uniform(self, lo, hi, *shape, dtype=torch.float32):
        return torch.empty(shape, dtype=torch.float32, device=DEV).uniform_(lo, hi, generator=self.g).to(dtype)

    def ints(self, lo, hi, *shape, dtype=torch.int8):
        """uniform in [lo, hi]"""
        return torch.empty(shape, dtype=dtype, device=DEV).random_(lo, hi + 1, generator=self.g)

    def mx_operand(self, fmt, rows, k):
        """normally distributed 8-bit floats, or uniformly distributed 4-bit codes"""
        if fmt == "e4m3":
            return self.normal(rows, k).to(torch.float8_e4m3fn).view(torch.uint8)
        if fmt == "e5m2":
            return self.normal(rows, k).to(torch.float8_e5m2).view(torch.uint8)
        return self.ints(0, 255, rows, k // 2, dtype=torch.uint8)


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, _Source(seed))


def run(state):
    return state["call"]()


def _prepare_quant(c, s):
    m, n, dt = c["m"], c["n"], FLOATS[c["src"]]
    x = s.normal(m, n, dtype=dt, std=2.0)
    codes = {"i8": torch.int8, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
    if c["policy"] == "dynamic":
        q, ts = torch.empty(m, n, dtype=torch.int8, device=DEV), torch.empty(m, dtype=torch.float32, device=DEV)
        return {"call": lambda: ops.dynamic_quant_per_token(x, q, ts)}
    dst = torch.empty(m, n // 2, dtype=torch.uint8, device=DEV) if c["dst"] == "e2m1" else torch.empty(m, n, dtype=codes[c["dst"]], device=DEV)
    top = {"i8": 127.0, "e4m3": 448.0, "e5m2": 57344.0, "e2m1": 6.0}[c["dst"]]
    if c["policy"] == "tensor":
        return {"call": lambda: ops.ascend_quant(dst, x, 15.0, 0.0)}
    if c["policy"] == "channel":
        scale = (127.0 / x.float().abs().amax(0).clamp_(min=0.5)).to(dt)
        return {"call": lambda: ops.ascend_quant(dst, x, scale, 0.0)}
    para = ops.AscendQuantParam(m=m, n=n, cal_count=m * n, group_size=128)
    if c["policy"] == "token":
        scale, policy = (top / x.float().abs().amax(1).clamp_(min=0.5)).contiguous(), abi.PER_TOKEN
    else:
        scale, policy = top / 8.0 * s.uniform(0.8, 1.2, m, (n + 127) // 128), abi.PER_GROUP
    fmt = abi.QDST_FP4_E2M1 if c["dst"] == "e2m1" else None
    return {"call": lambda: ops.ascend_quant_policy(dst, x, scale, None, para, policy, dst_format=fmt)}


def _prepare_dequant(c, s):
    m, n, dt = c["m"], c["n"], FLOATS[c["dst"]]
    acc = s.ints(-2 ** 20, 2 ** 20, m, n, dtype=torch.int32)
    dst = torch.zeros(m, ops.dequant_dst_stride(dt, n), dtype=dt, device=DEV)
    if c["policy"] in ("channel", "tensor"):
        scale = s.uniform(1e-5, 1e-3, n) if c["policy"] == "channel" else 1e-4
        para = ops.DequantParams(m=m, n=n, cal_count=n)
        return {"call": lambda: ops.ascend_dequant(dst, acc, scale, para)}
    para = ops.AscendQuantParam(m=m, n=n, cal_count=m * n, group_size=128)
    token = c["policy"] == "token"
    scale = s.uniform(1e-5, 1e-3, m) if token else s.uniform(1e-5, 1e-3, m, (n + 127) // 128)
    policy = abi.PER_TOKEN if token else abi.PER_GROUP
    return {"call": lambda: ops.ascend_dequant_policy(dst, acc, scale, para, policy)}


def _prepare_antiquant(c, s):
    m, n, dt, g = c["m"], c["n"], FLOATS[c["dst"]], c["groups"]
    dst = torch.empty(m, n, dtype=dt, device=DEV)
    if c["src"] in ("i8", "i4"):
        src = s.ints(-128, 127, m, n) if c["src"] == "i8" else s.ints(0, 255, m, n // 2, dtype=torch.uint8)
        shape = (m, g) if c["transposed"] else (g, n)
        scale = s.uniform(1e-3, 1e-2, *shape, dtype=dt)
        offset = s.uniform(-8.0, 8.0, *shape, dtype=dt) if c["offset"] else None
        info = ops.AntiQuantShapeInfo(shape[0], shape[1], shape[0], shape[1])
        k, int4 = (n if c["transposed"] else m), c["src"] == "i4"
        return {"call": lambda: ops.ascend_antiquant(dst, src, offset, scale, k, info, c["transposed"], int4)}
    para = ops.AscendAntiQuantParam(m=m, n=n, cal_count=m * n, group_size=128)
    if c["src"] == "e2m1":
        src = s.mx_operand("e2m1", m, n)
        scale = s.ints(121, 127, m, (n + 127) // 128, dtype=torch.uint8)
        return {"call": lambda: ops.ascend_antiquant_policy(dst, src, scale, None, para, abi.PER_GROUP, src_format=abi.QDST_FP4_E2M1)}
    src = s.normal(m, n).to(torch.float8_e4m3fn)
    shape, policy = ((m,), abi.PER_TOKEN) if g == 1 else ((m, (n + 127) // 128), abi.PER_GROUP)
    scale = s.uniform(1e-2, 1e-1, *shape)
    offset = s.uniform(-1.0, 1.0, *shape) if c["offset"] else None
    config = ops.AscendAntiQuantConfig(has_offset=c["offset"])
    config.k_dim = 1
    return {"call": lambda: ops.ascend_antiquant_policy(dst, src, scale, offset, para, policy, config)}


def _bias(s, which, *shape):
    return None if which == "none" else s.normal(*shape, dtype=FLOATS[which])


def _prepare_linear(c, s):
    m, k, n, dt = c["m"], c["k"], c["n"], FLOATS[c["x"]]
    x = s.normal(m, k, dtype=dt)
    nk = c["weights"] == "nk"
    w = s.ints(-127, 127, *((n, k) if nk else (k, n)))
    cs = s.uniform(1e-4, 1e-3, n)
    bias = _bias(s, c["bias"], n)
    out = torch.empty(m, n // 2 if c["act"] == "swiglu" else n, dtype=FLOATS[c["out"]], device=DEV)
    packed = c["weights"] == "packed"
    if packed:
        w = ops.pack_weight_w8(w, k, n)
    act = ACT[c["act"]]
    if m <= 64:
        # decode: the same few rows step after step, through a handle made once
        lin = ops.DynamicLinear(m, k, w, cs, bias, trans_b=nk, packed_n=n if packed else None, out_dtype=FLOATS[c["out"]], x_dtype=dt,
                                activation=act)
        return {"call": lambda: lin(out, x)}
    if packed:
        return {"call": lambda: ops.linear_w8a8_dynamic_packed(out, x, w, n, cs, bias, act)}
    return {"call": lambda: ops.linear_w8a8_dynamic(out, x, w, cs, bias, act, nk)}


def _prepare_w4a16(c, s):
    m, k, n, g = c["m"], c["k"], c["n"], c["group"]
    x = s.normal(m, k, dtype=torch.float16)
    w = s.ints(0, 255, k, n // 2, dtype=torch.uint8)
    scale = s.uniform(1e-3, 1e-2, k // g, n, dtype=torch.float16)
    offset = s.uniform(-8.0, 8.0, k // g, n, dtype=torch.float16) if c["offset"] else None
    y = torch.empty(m, n, dtype=torch.float16, device=DEV)
    if c["weights"] == "nd":
        return {"call": lambda: ops.matmul_w4a16(y, x, w, scale, offset, g)}
    w = ops.pack_weight_w4(w, k, n)
    mode = abi.W4A16_GROUP_SUM if c["mode"] == "group_sum" else abi.W4A16_PER_WEIGHT
    return {"call": lambda: ops.matmul_w4a16_packed(y, x, w, scale, offset, g, mode)}


def _prepare_w8a16(c, s):
    m, k, n = c["m"], c["k"], c["n"]
    x = s.normal(m, k, dtype=torch.float16)
    nk = c["weights"] == "nk"
    w = s.ints(-127, 127, *((n, k) if nk else (k, n)))
    if c["per_tensor"]:
        scale, offset = 3e-3, 1.5 if c["offset"] else None
    else:
        scale = s.uniform(1e-3, 1e-2, n, dtype=torch.float16)
        offset = s.uniform(-8.0, 8.0, n, dtype=torch.float16) if c["offset"] else None
    y = torch.empty(m, n, dtype=FLOATS[c["out"]], device=DEV)
    mode = 1 if c["mode"] == "channel_sum" else abi.W8A16_PER_WEIGHT
    return {"call": lambda: ops.matmul_w8a16(y, x, w, offset, scale, trans_b=nk, mode=mode)}


def _prepare_moe(c, s):
    g, m, k, n = c["groups"], c["tokens"], c["k"], c["n"]
    x = s.ints(-127, 127, m, k)
    w = s.ints(-127, 127, g, k, n)
    if c["weights"] == "nz":
        w = ops.pack_weight_nz(w)
    scale = s.uniform(1e-4, 1e-3, g, n)
    tok = s.uniform(5e-3, 2e-2, m)
    bias = _bias(s, c["bias"], g, n)
    # tokens per expert: a multinomial draw, with `skew` some experts are more popular than others
    popularity = torch.exp(c["skew"] * s.normal(g))
    picks = torch.multinomial(popularity, m, replacement=True, generator=s.g)
    counts = torch.bincount(picks, minlength=g).to(torch.int64)
    y = torch.empty(m, n // 2 if c["act"] == "swiglu" else n, dtype=FLOATS[c["out"]], device=DEV)
    return {"call": lambda: ops.quant_group_matmul(y, x, w, counts, scale, tok, bias, activation=ACT[c["act"]],
                                                   weight_nz=c["weights"] == "nz")}


def _prepare_mx(c, s):
    m, n, k = c["m"], c["n"], c["k"]
    a, b = s.mx_operand(c["a"], m, k), s.mx_operand(c["b"], n, k)
    sk = (k // 32 + 7) // 8 * 8
    sa, sb = s.ints(123, 129, m, sk, dtype=torch.uint8), s.ints(119, 125, n, sk, dtype=torch.uint8)
    bias = s.normal(n) if c["bias"] else None
    y = torch.empty(m, n, dtype=FLOATS[c["out"]], device=DEV)
    return {"call": lambda: ops.matmul_mx(y, a, b, sa, sb, MX_FORMAT[c["a"]], MX_FORMAT[c["b"]], k, bias)}


# ------------------------------------------------------------------------------------------------- work, tolerances
def work(case):
    c, kind = case, case["kind"]
    if kind in ("quant", "dequant", "antiquant"):
        m, n = c["m"], c["n"]
        size_in = SIZE[c["src"]] if kind != "dequant" else 4
        if kind == "antiquant" and c["src"] in ("i8", "i4"):
            params = (m if c["transposed"] else n) * c["groups"] * SIZE[c["dst"]] * (2 if c["offset"] else 1)
        elif kind == "antiquant":
            params = m * (1 if c["groups"] == 1 and c["src"] != "e2m1" else (n + 127) // 128) * (1 if c["src"] == "e2m1" else 4)
            params *= 2 if c["offset"] else 1
        else:
            params = {"channel": n * (SIZE[c["src"]] if kind == "quant" else 4), "tensor": 0, "token": m * 4, "dynamic": m * 4,
                      "group": m * ((n + 127) // 128) * 4}[c["policy"]]
        return {"bytes": int(m * n * (size_in + SIZE[c["dst"]]) + params), "flops": 2 * m * n}
    k, n = c["k"], c["n"]
    m = c["tokens"] if kind == "moe" else c["m"]
    cols = n // 2 if c.get("act") == "swiglu" else n
    flops = 2 * m * n * k
    if kind == "linear":
        return {"bytes": m * k * 2 + k * n + n * 4 + m * cols * 2 + (0 if c["bias"] == "none" else n * SIZE[c["bias"]]), "flops": flops}
    if kind == "w4a16":
        return {"bytes": m * k * 2 + k * n // 2 + k // c["group"] * n * (4 if c["offset"] else 2) + m * n * 2, "flops": flops}
    if kind == "w8a16":
        return {"bytes": m * k * 2 + k * n + (0 if c["per_tensor"] else n * (4 if c["offset"] else 2)) + m * n * SIZE[c["out"]],
                "flops": flops}
    if kind == "moe":
        # experts that no token went to need not be read
        busy = min(c["groups"], m)
        return {"bytes": m * k + busy * k * n + busy * n * (4 + (2 if c["bias"] == "bf16" else 0)) + m * 4 + m * cols * 2, "flops": flops}
    return {"bytes": int(m * k * SIZE[c["a"]] + n * k * SIZE[c["b"]] + (m + n) * (k // 32) + m * n * SIZE[c["out"]]), "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("quant", "dequant", "antiquant"):
        return "exact"      # every rounding of these operators is specified
    # outputs rounded once to 8 (bf16) or 11 (f16) significant bits: 1.7e-3 and 2.1e-4 of the result (2-norm) measured
    # against the same product in 64 bits; fp32 outputs carry the order of their sums
    out = {"bf16": 7e-3, "f16": 9e-4, "f32": 2e-5}[case.get("out", "f16")]
    if kind == "w4a16" or kind == "w8a16":
        # weights rounded to half twice, or not at all: 3.7e-4 between the two forms of the same product
        return {"rel": 1.5e-3}
    if kind == "linear":
        # a quantised activation may land on the other side of a tie: 4.8e-4 (6.6e-4 with SwiGLU) on half outputs
        return {"rel": max(out, 2.5e-3)}
    if kind == "mx" and "e4m3" in (case["a"], case["b"]):
        # the matrix core aligns the products of a block of 8-bit operands before it adds them: 1.4e-5
        return {"rel": max(out, 6e-5)}
    return {"rel": out}
