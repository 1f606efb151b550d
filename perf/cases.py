"""The framework's calls that its performance is measured on.

Each case is one call (or the short sequence of calls that belong together) that a
serving engine makes through the public operators: dense W4A16 linears from decode
to prefill, the routed MoE layer over the same range, the routed grouped GEMM under
both of its entry points, and the W4A4 path with its activation quantizer.  The
shapes are those of bench.py and the tests (qkv_proj 2048 -> 5120, o_proj
4096 -> 2048, 128 experts, top-8, hidden 2048, intermediate 768); ``draw`` spreads
the same calls over generic sizes.  Weight codes are uniform over the 16 E2M1
codes with E8M0 bytes uniform in 120..128 and activations N(0, 1), as in bench.py.
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "mxfp4-gfx936_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mxfp4_amd as mx  # noqa: E402

_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32,
       "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4, "e4m3": 1, "e5m2": 1, "mxfp4": 17 / 32}
_W = 17 / 32  # bytes of one MXFP4 weight with its share of the E8M0 byte


def listed():
    moe = {"e": 128, "top_k": 8, "h": 2048, "i": 768}
    return [
        # one token through a qkv projection: the smallest call, where the launch
        # and the host path count; the weights were prepacked at load, as the
        # vLLM hooks do
        {"name": "linear_m1", "op": "linear", "m": 1, "k": 2048, "n": 5120, "x": "bf16",
         "bias": False, "pre": True},
        # a batch of decode requests through an output projection with a bias
        {"name": "linear_m64_fp16", "op": "linear", "m": 64, "k": 4096, "n": 2048, "x": "fp16",
         "bias": True, "pre": True},
        # a ragged prompt chunk through o_proj on the checkpoint layout (the
        # reference's signature, no copy registered)
        {"name": "linear_m370", "op": "linear", "m": 370, "k": 4096, "n": 2048, "x": "bf16",
         "bias": False, "pre": False},
        # prefill of a full chunk through qkv_proj (the headline workload)
        {"name": "linear_m4096", "op": "linear", "m": 4096, "k": 2048, "n": 5120, "x": "bf16",
         "bias": False, "pre": True},
        # one token through the routed MoE layer
        {"name": "moe_m1", "op": "moe", "m": 1, **moe, "x": "bf16", "pre": True,
         "router": False},
        # a decode step as an engine runs it: qkv and output projections, router
        # and MoE layer of one block for 8 requests, captured once in a HIP graph
        # and replayed
        {"name": "decode_graph_m8", "op": "decode", "m": 8, **moe, "qkv": 5120, "o": 4096,
         "x": "bf16", "pre": True},
        # a larger decode batch through the MoE layer
        {"name": "moe_m32", "op": "moe", "m": 32, **moe, "x": "bf16", "pre": True,
         "router": False},
        # a prompt chunk through router and MoE layer
        {"name": "moe_m512_router", "op": "moe", "m": 512, **moe, "x": "bf16", "pre": True,
         "router": True},
        # full prefill through the MoE layer: the largest call
        {"name": "moe_m4096", "op": "moe", "m": 4096, **moe, "x": "bf16", "pre": True,
         "router": False},
        # the drop-in routed GEMM (gate_up) on the checkpoint layout, odd token count
        {"name": "soft_m509", "op": "soft", "m": 509, "e": 128, "top_k": 8, "k": 2048, "n": 1536,
         "a": "bf16", "c": "bf16", "weighted": False},
        # AITER's entry with FP8 activations on the caller's routing metadata
        # (down projection with route weights)
        {"name": "aiter_fp8_m1000", "op": "aiter", "m": 1000, "e": 128, "top_k": 8, "k": 768,
         "n": 2048, "a": "e4m3", "c": "bf16", "weighted": True, "block_m": 64},
        # W4A4: activation quantizer and dense GEMM on the block-scaled MFMA
        {"name": "w4a4_m8192", "op": "w4a4", "m": 8192, "k": 4096, "n": 4096, "x": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_MOST_MACS = 4096 * 8 * 3 * 2048 * 768  # of the largest listed case
_MOST_WEIGHTS = 128 * 3 * 2048 * 768


def _fit_moe(e, macs_per_token, weights_per_expert, m):
    """Experts and tokens of a drawn routed case within the largest listed one."""
    while e > 8 and e * weights_per_expert > _MOST_WEIGHTS:
        e //= 2
    return e, max(1, min(m, _MOST_MACS // macs_per_token))


def draw(rng):
    op = rng.choice(["linear", "linear", "linear", "moe", "moe", "moe", "decode", "soft", "aiter",
                     "w4a4"])
    if op == "linear":
        n = _log_int(rng, 512, 6144)
        # mostly whole tiles of 64; some sharded or padded widths
        n = n // 8 * 8 if rng.random() < 0.25 else max(512, n // 64 * 64)
        return {"op": op, "m": _log_int(rng, 1, 4096), "k": 128 * _log_int(rng, 4, 36), "n": n,
                "x": rng.choice(["bf16", "bf16", "fp16"]), "bias": rng.random() < 0.3,
                "pre": rng.random() < 0.6}
    if op == "w4a4":
        return {"op": op, "m": _log_int(rng, 16, 8192), "k": 128 * _log_int(rng, 8, 32),
                "n": 64 * _log_int(rng, 8, 64), "x": rng.choice(["bf16", "bf16", "fp16"])}
    e, top_k = rng.choice([(8, 2), (32, 4), (64, 6), (128, 8), (128, 8)])
    if op in ("moe", "decode"):
        h, i = rng.choice([1024, 2048, 2048, 2880, 4096]), rng.choice([512, 768, 1024, 1408])
        m = _log_int(rng, 1, 64 if op == "decode" else 4096)
        e, m = _fit_moe(e, top_k * 3 * h * i, 3 * h * i, m)
        case = {"op": op, "m": m, "e": e, "top_k": min(top_k, e), "h": h, "i": i, "x": "bf16",
                "pre": rng.random() < 0.7}
        if op == "moe":
            case["router"] = rng.random() < 0.4
        else:
            case["qkv"], case["o"] = 128 * _log_int(rng, 8, 48), 128 * _log_int(rng, 8, 32)
            if h % 128:  # the dense linear's K
                case["h"] = 2048
                case["e"], case["m"] = _fit_moe(e, top_k * 3 * 2048 * i, 3 * 2048 * i, m)
                case["top_k"] = min(top_k, case["e"])
        return case
    k, n = rng.choice([768, 1024, 2048, 2048, 4096]), rng.choice([1024, 1536, 1536, 2048, 4096])
    e, m = _fit_moe(e, top_k * k * n, k * n, _log_int(rng, 1, 4096))
    case = {"op": op, "m": m, "e": e, "top_k": min(top_k, e), "k": k, "n": n,
            "weighted": rng.random() < 0.5}
    if op == "soft":
        case["a"] = rng.choice(["bf16", "bf16", "fp16", "mxfp4"])
        case["c"] = "fp16" if case["a"] == "fp16" else rng.choice(["bf16", "bf16", "fp32"])
        if case["c"] == "fp32":
            case["m"] = min(case["m"], 1024)
    else:
        case["a"] = rng.choice(["bf16", "e4m3", "e5m2", "mxfp4"])
        case["c"], case["block_m"] = "bf16", rng.choice([32, 64, 128])
    return case


# ------------------------------------------------------------------- inputs

def _weights(gen, *shape):
    """Packed codes [..., N, K/2] and E8M0 bytes [..., N, K/32] for [..., N, K]."""
    *lead, k = shape
    p = torch.randint(0, 256, (*lead, k // 2), generator=gen, device="cuda", dtype=torch.uint8)
    s = torch.randint(120, 129, (*lead, k // 32), generator=gen, device="cuda", dtype=torch.uint8)
    return p, s


def _act(gen, dtype, *shape):
    return torch.randn(shape, generator=gen, device="cuda").to(_DT[dtype])


def _quant_rne(x):
    """OCP MX quantization of [..., K] in plain torch: E = floor(log2(amax)) - 2
    per 32, E2M1 with ties to the even code, saturating; (packed, scales)."""
    b = x.double().reshape(*x.shape[:-1], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    _, e = torch.frexp(amax)
    e = torch.where(amax == 0, torch.full_like(e, -127), e - 3).clamp(-127, 127)
    q = torch.ldexp(b, -e)
    a = q.abs()
    r = torch.where(a < 2, torch.round(a * 2) / 2,
                    torch.where(a < 4, torch.round(a), torch.round(a / 2) * 2)).clamp(max=6)
    code = torch.where(r < 2, r * 2, torch.where(r < 4, r + 2, r / 2 + 4)).to(torch.uint8)
    code = code | (torch.signbit(q).to(torch.uint8) << 3)
    code = code.reshape(*x.shape[:-1], -1, 2)
    packed = code[..., 0] | (code[..., 1] << 4)
    return packed, (e[..., 0] + 127).to(torch.uint8)


def _route(logits, top_k):
    """softmax -> top-k -> renormalize, as the reference's tests route."""
    w, ids = torch.topk(torch.softmax(logits, -1), top_k, dim=-1)
    return w / w.sum(-1, keepdim=True), ids


def _inputs(case, seed):
    """The tensors of a case: a function of the case and the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    op, m = case["op"], case["m"]
    t = {}
    if op == "linear":
        t["w"], t["ws"] = _weights(g, case["n"], case["k"])
        t["x"] = _act(g, case["x"], m, case["k"])
        t["bias"] = _act(g, case["x"], case["n"]) if case["bias"] else None
    elif op in ("moe", "decode"):
        e, h, i = case["e"], case["h"], case["i"]
        t["w13"], t["s13"] = _weights(g, e, 2 * i, h)
        t["w2"], t["s2"] = _weights(g, e, h, i)
        t["x"] = _act(g, case["x"], m, h)
        t["logits"] = _act(g, "fp32", m, e)
        if op == "decode":
            t["wq"], t["sq"] = _weights(g, case["qkv"], h)
            t["wo"], t["so"] = _weights(g, h, case["o"])
            t["attn"] = _act(g, case["x"], m, case["o"])
        elif not case["router"]:
            t["tw"], t["ids"] = _route(t["logits"], case["top_k"])
    elif op in ("soft", "aiter"):
        e, k, n = case["e"], case["k"], case["n"]
        t["w"], t["ws"] = _weights(g, e, n, k)
        t["tw"], t["ids"] = _route(_act(g, "fp32", m, e), case["top_k"])
        t["a_scale"] = torch.full((1,), 0.75, device="cuda")
        t["b_scale"] = 0.5 + torch.rand(e, generator=g, device="cuda")
        if case["a"] == "mxfp4":
            t["a"], t["a_mx"] = _quant_rne(_act(g, "bf16", m, k))
        else:
            t["a"], t["a_mx"] = _act(g, case["a"], m, k), None
    else:
        t["x"] = _act(g, case["x"], m, case["k"])
        t["w"], t["ws"] = _quant_rne(0.02 * _act(g, "fp32", case["n"], case["k"]))
    return t


# ------------------------------------------------------------- the measured call

def _decode_block(s):
    """One block of a decode step; attention itself is the engine's own."""
    qkv = mx.linear_mxfp4_soft(s["x"], s["wq"], s["sq"], prepacked=s["preq"])
    o = mx.linear_mxfp4_soft(s["attn"], s["wo"], s["so"], prepacked=s["preo"])
    tw, ids = mx.route_topk(s["logits"], s["top_k"])
    y = mx.moe_layer(s["x"], s["w13"], s["s13"], s["w2"], s["s2"], tw, ids,
                     prepacked13=s["pre13"], prepacked2=s["pre2"])
    return {"qkv": qkv, "o": o, "tw": tw, "ids": ids, "y": y}


def prepare(case, seed):
    s = _inputs(case, seed)
    op = case["op"]
    s["op"] = op
    pack = mx.prepack_w4a16 if case.get("pre") else lambda p, sc: None
    if op == "linear":
        s["pre"] = pack(s["w"], s["ws"])
    elif op in ("moe", "decode"):
        s["pre13"], s["pre2"] = pack(s["w13"], s["s13"]), pack(s["w2"], s["s2"])
        s["top_k"] = case["top_k"]
        s["router"] = case.get("router", True)
        if op == "decode":
            s["preq"], s["preo"] = pack(s["wq"], s["sq"]), pack(s["wo"], s["so"])
            _decode_block(s)  # once outside the capture
            torch.cuda.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                s["out"] = _decode_block(s)
    elif op in ("soft", "aiter"):
        s["c"] = torch.zeros((case["m"], case["top_k"], case["n"]), dtype=_DT[case["c"]],
                             device="cuda")
        s["top_k"], s["weighted"], s["e"] = case["top_k"], case["weighted"], case["e"]
        s["none"] = torch.empty(0, dtype=torch.int32, device="cuda")
        s["block_m"] = case.get("block_m")
        s["config"] = {"BLOCK_SIZE_M": s["block_m"]}
    return s


def run(s):
    op = s["op"]
    if op == "linear":
        return mx.linear_mxfp4_soft(s["x"], s["w"], s["ws"], s["bias"], prepacked=s["pre"])
    if op == "moe":
        if not s["router"]:
            return mx.moe_layer(s["x"], s["w13"], s["s13"], s["w2"], s["s2"], s["tw"], s["ids"],
                                prepacked13=s["pre13"], prepacked2=s["pre2"])
        tw, ids = mx.route_topk(s["logits"], s["top_k"])
        y = mx.moe_layer(s["x"], s["w13"], s["s13"], s["w2"], s["s2"], tw, ids,
                         prepacked13=s["pre13"], prepacked2=s["pre2"])
        return {"tw": tw, "ids": ids, "y": y}
    if op == "decode":
        s["graph"].replay()
        return s["out"]
    if op == "soft":
        # the safe operator builds its routing itself
        mx.fused_moe_mxfp4_soft(s["a"], s["w"], s["c"], s["a_scale"], s["b_scale"], s["a_mx"],
                                s["ws"], s["tw"], s["ids"], s["none"], s["none"], s["none"],
                                s["weighted"], s["top_k"], False, False)
        return s["c"]
    if op == "aiter":
        sorted_ids, expert_ids, npp = mx.make_routing(s["ids"], s["block_m"], s["e"])
        mx.fused_moe_mxfp4(s["a"], s["w"], s["c"], s["a_scale"], s["b_scale"], s["a_mx"], s["ws"],
                           s["tw"], s["ids"], sorted_ids, expert_ids, npp, s["weighted"],
                           s["top_k"], False, False, s["config"], s["c"].dtype)
        return s["c"]
    packed, scales = mx.dynamic_mxfp4_quant(s["x"], mode="rne")
    return {"packed": packed, "scales": scales,
            "y": mx.linear_mxfp4_w4a4(packed, scales, s["w"], s["ws"])}


# -------------------------------------------------------------- what it takes

def _active(case):
    """Experts that uniform routing is expected to touch."""
    e = case["e"]
    return e * (1 - (1 - case["top_k"] / e) ** case["m"])


def work(case):
    op, m = case["op"], case["m"]
    if op == "linear":
        k, n, b = case["k"], case["n"], _BYTES[case["x"]]
        return {"bytes": n * k * _W + m * (k + n) * b + (n * b if case["bias"] else 0),
                "flops": 2 * m * n * k}
    if op == "w4a4":
        k, n = case["k"], case["n"]
        return {"bytes": n * k * _W + m * k * (2 + _W) + m * n * 2, "flops": 2 * m * n * k}
    r = m * case["top_k"]
    if op in ("moe", "decode"):
        h, i = case["h"], case["i"]
        nbytes = _active(case) * 3 * h * i * _W + 2 * m * h * 2 + r * 12
        flops = 2 * r * 3 * h * i
        if op == "decode" or case["router"]:
            nbytes += m * case["e"] * 4
        if op == "decode":
            q, o = case["qkv"], case["o"]
            nbytes += (q * h + h * o) * _W + m * (q + h + o) * 2
            flops += 2 * m * (q * h + h * o)
        return {"bytes": nbytes, "flops": flops}
    k, n = case["k"], case["n"]
    return {"bytes": _active(case) * k * n * _W + m * k * _BYTES[case["a"]]
            + r * n * _BYTES[case["c"]] + r * 12, "flops": 2 * r * n * k}


def tolerance(case):
    """About four times the distance measured from the 64-bit result."""
    if case["op"] in ("moe", "decode"):
        # gate, up, silu and their product are rounded to bf16 between the GEMMs:
        # measured rel 0.0038, max 0.027
        return {"rel": 0.015, "max": 0.1}
    if case["op"] == "soft" and case["c"] == "fp32":
        # sums over K: measured rel 2.3e-7, max 1.8e-6
        return {"rel": 1e-6, "max": 8e-6}
    if case["op"] != "w4a4" and case.get("c", case.get("x")) == "fp16":
        return {"rel": 8e-4, "max": 2e-3}  # one rounding to fp16: rel 2.1e-4, max 4.9e-4
    return {"rel": 7e-3, "max": 0.016}  # one rounding to bf16: rel 1.7e-3, max 3.9e-3


# ------------------------------------------------------- the same in 64 bits

_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _dequant64(packed, scales):
    lut = torch.tensor(_E2M1, dtype=torch.float64, device=packed.device)
    codes = torch.stack([packed & 15, packed >> 4], -1).reshape(*packed.shape[:-1], -1)
    v = lut[codes.int()].reshape(*scales.shape, 32)
    return torch.ldexp(v, scales.int().sub(127).unsqueeze(-1)).reshape(codes.shape)


def _moe64(t, w, ids):
    x, i = t["x"].double(), t["w13"].shape[1] // 2
    y = torch.zeros_like(x)
    for e in range(t["w13"].shape[0]):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        gu = x[tok] @ _dequant64(t["w13"][e], t["s13"][e]).T
        hid = torch.nn.functional.silu(gu[:, :i]) * gu[:, i:]
        down = hid @ _dequant64(t["w2"][e], t["s2"][e]).T
        y.index_add_(0, tok, down * w[tok, slot].double().unsqueeze(-1))
    return y


def exact(case, seed):
    t = _inputs(case, seed)
    op = case["op"]
    if op == "linear":
        y = t["x"].double() @ _dequant64(t["w"], t["ws"]).T
        return y if t["bias"] is None else y + t["bias"].double()
    if op == "w4a4":
        packed, scales = _quant_rne(t["x"])
        return {"packed": packed, "scales": scales,
                "y": _dequant64(packed, scales) @ _dequant64(t["w"], t["ws"]).T}
    if op in ("moe", "decode"):
        if op == "moe" and not case["router"]:
            return _moe64(t, t["tw"], t["ids"])
        w, ids = _route(t["logits"].double(), case["top_k"])
        out = {"tw": w, "ids": ids, "y": _moe64(t, w, ids)}
        if op == "decode":
            out["qkv"] = t["x"].double() @ _dequant64(t["wq"], t["sq"]).T
            out["o"] = t["attn"].double() @ _dequant64(t["wo"], t["so"]).T
        return out
    a = _dequant64(t["a"], t["a_mx"]) if case["a"] == "mxfp4" else t["a"].double()
    c = torch.zeros((case["m"], case["top_k"], case["n"]), dtype=torch.float64, device="cuda")
    for e in range(case["e"]):
        tok, slot = torch.nonzero(t["ids"] == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        v = a[tok] @ _dequant64(t["w"][e], t["ws"][e]).T
        v = v * (t["a_scale"][0].double() * t["b_scale"][e].double())
        if case["weighted"]:
            v = v * t["tw"][tok, slot].double().unsqueeze(-1)
        c[tok, slot] = v
    return c
