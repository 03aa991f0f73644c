"""The work this framework is measured on: what a serving program has it do around every GEMM.

Each case is one pass through the public operators (`mcoplib.op`, `mcoplib.custom_ops` and
`torch.ops._C`) on tensors that the program already holds on the GPU: activations (the output of
the GEMM before), the running residual, the layer's weight and, for SmoothQuant, its smooth
scales.  `calls` > 1 stands for the same operator in consecutive layers (each with inputs and a
weight of its own, all on one running residual); `graph` for a pass captured once and replayed,
as servers run their decode steps.

Activations are N(0, 1) with 1% of the channels scaled by 20 (the outlier channels that per-token
quantization meets in earnest), weights N(1, 0.1), smooth scales U(0.5, 2).
"""

from __future__ import annotations

import math

import torch

import mcoplib._C  # noqa: F401  (registers torch.ops._C)
from mcoplib import custom_ops, op

EPS = 1e-6
GROUP = 128  # elements per scale of the per-block quantizer
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
QUANT = {"int8": torch.int8, "fp8": torch.float8_e4m3fn}


def _case(op, tokens, hidden, dtype="bf16", quant="int8", residual=True, bound=False, calls=1,
          graph=False, **more):
    return dict(op=op, tokens=tokens, hidden=hidden, dtype=dtype, quant=quant, residual=residual,
                bound=bound, calls=calls, graph=graph, **more)


def listed():
    return [
        # one token of one user: the two norms of one layer, called eagerly (smallest call there is)
        dict(name="decode_t1", **_case("add_norm_int8", 1, 5120, calls=2)),
        # a decode step of 64 sequences: the norms of an 8-layer stack, replayed from a graph
        dict(name="decode_t64_graph", **_case("add_norm_int8", 64, 5120, calls=16, graph=True)),
        # prefill of 8192 tokens at a 70B-class width, int8 weights and activations (W8A8)
        dict(name="prefill_int8", **_case("add_norm_int8", 8192, 8192)),
        # the largest: 32k tokens in one batch at the widest hidden size in the configurations
        dict(name="prefill_int8_large", **_case("add_norm_int8", 32768, 16384)),
        # vLLM's operator with fp8 codes at the odd width of its own test suite
        dict(name="norm_fp8_ragged", **_case("norm_quant", 2048, 5137, quant="fp8")),
        # an unquantized layer: residual add + RMSNorm, both in place
        dict(name="fused_add_norm", **_case("fused_add_norm", 4096, 4096)),
        # SmoothQuant with fp8 codes, after_res and after_norm kept: 16k tokens at width 7168
        dict(name="smooth_fp8", **_case("smooth", 16384, 7168, quant="fp8", residual=False)),
        # the same operator on rows far wider than one workgroup's registers
        dict(name="smooth_fp8_wide", **_case("smooth", 2048, 131072, quant="fp8",
                                             residual=False)),
        # activation quantizer before an fp8 GEMM, on one half of a fused projection's output
        # (rows strided)
        dict(name="token_fp8_strided", **_case("token_fp8", 4096, 8192, quant="fp8",
                                               residual=False, strided=True)),
        # expert-parallel dispatch: codes and scale of a token packed into one padded row
        dict(name="padded_dispatch", **_case("padded", 2048, 7168)),
        # block-scaled fp8 (one scale per 128 channels), for block-scaled GEMMs
        dict(name="block_fp8", **_case("block_quant", 8192, 8192, quant="fp8",
                                       transposed=False)),
        # q/k norm: 8 heads of 128 for 16k tokens
        dict(name="head_norm", **_case("head_norm", 16384, 128, residual=False, heads=8)),
    ]


OPS = ("add_norm_int8", "norm_quant", "fused_add_norm", "smooth", "scale_quant", "token_int8",
       "token_int8_azp", "token_fp8", "padded", "block_quant", "norm", "vllm_norm", "head_norm")
MOST_ELEMENTS = 1 << 28  # of a drawn case: below the largest listed one's 2^29


def draw(rng):
    """Any operator; 1 to 32768 tokens; rows of 64 to 131072 elements, one third of them odd."""
    name = rng.choice(OPS)
    hidden = int(2 ** rng.uniform(6, 17))
    if name == "block_quant":
        hidden = max(1, hidden // GROUP) * GROUP
    elif rng.random() < 1 / 3:
        hidden |= 1
    else:
        hidden = hidden // 64 * 64
    more = {}
    if name == "head_norm":
        hidden, more["heads"] = rng.choice((64, 80, 96, 128, 192, 256)), rng.randint(1, 32)
    row = hidden * more.get("heads", 1)
    tokens = int(2 ** rng.uniform(0, min(15, math.log2(MOST_ELEMENTS / row))))
    only_bf16 = name in ("padded", "scale_quant")
    dtype = "bf16" if only_bf16 else rng.choice(("bf16",) * 4 + ("fp16", "fp32"))
    if name == "head_norm" and dtype == "fp16":
        dtype = "fp32"  # its weights are bf16 or fp32
    quant = "fp8" if name == "token_fp8" or (name in ("norm_quant", "smooth", "block_quant")
                                             and rng.random() < 0.5) else "int8"
    residual = name in ("add_norm_int8", "fused_add_norm", "padded") or (
        name in ("norm_quant", "smooth", "block_quant", "norm") and rng.random() < 0.6)
    bound = name in ("norm_quant", "token_fp8") and rng.random() < 0.2
    if name == "block_quant":
        more["transposed"] = rng.random() < 0.5
    if name == "token_fp8":
        more["strided"] = rng.random() < 0.3
    # small calls come as a stack of layers; decode steps from a graph half of the time
    calls = 8 if tokens * row < 1 << 20 else 1
    graph = calls > 1 and rng.random() < 0.5 and hidden <= 32768
    return _case(name, tokens, hidden, dtype, quant, residual, bound, calls, graph, **more)


# ------------------------------------------------------------------------------------- inputs
def _inputs(case, seed):
    """x [calls, tokens, hidden] (heads: [calls, tokens, heads, hidden]), weights, the residual,
    smooth scales and the scale bound, from the seed alone."""
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    n, T, H, dt = case["calls"], case["tokens"], case["hidden"], DTYPES[case["dtype"]]
    heads = case.get("heads")
    shape = (n, T, heads, H) if heads else (n, T, H)
    wide = (*shape[:-1], 2 * H) if case.get("strided") else shape

    def normal(*s):
        return torch.empty(s, dtype=dt, device=dev).normal_(generator=g)

    x = normal(*wide)[..., :H]
    outliers = torch.randperm(H, generator=g, device=dev)[:round(0.01 * H)]
    x[..., outliers] *= 20
    i = {"x": x, "r": None, "sm": None, "ub": None}
    i["w"] = 1 + 0.1 * normal(*((n, heads, H) if heads else (n, H)))
    if case["residual"]:
        i["r"] = normal(T, H)
    if case["op"] in ("smooth", "scale_quant"):
        i["sm"] = 0.5 + 1.5 * torch.rand(n, H, generator=g, device=dev)
    if case["bound"]:
        i["ub"] = torch.full((1,), 4.0, device=dev)
    return i


def _pad_size(H):
    """bf16 elements of a padded row: the codes, the scale, and up to whole 64-byte lines."""
    return (H + 4 + 63) // 64 * 32


def prepare(case, seed):
    s = {**case, **_inputs(case, seed)}
    x, dev, T, H = s["x"], s["x"].device, case["tokens"], case["hidden"]
    q, out = QUANT[case["quant"]], []
    for k in range(case["calls"]):
        o = {}
        if case["op"] in ("norm_quant", "smooth", "block_quant", "token_int8", "token_int8_azp",
                          "token_fp8"):
            o["q"] = torch.empty(T, H, dtype=q, device=dev)
            o["s"] = torch.empty(T, 1, dtype=torch.float32, device=dev)
        if case["op"] == "block_quant":
            groups = (H // GROUP, T) if case["transposed"] else (T, H // GROUP)
            o["s"] = torch.empty(groups, dtype=torch.float32, device=dev)
        if case["op"] == "token_int8_azp":
            o["azp"] = torch.empty(T, 1, dtype=torch.int32, device=dev)
        if case["op"] == "smooth":
            o["after_res"], o["after_norm"] = torch.empty_like(x[k]), torch.empty_like(x[k])
        if case["op"] in ("norm", "vllm_norm", "head_norm"):
            o["out"] = torch.empty_like(x[k])
        if case["op"] == "norm":
            o["after_res"] = torch.empty_like(x[k]) if case["residual"] else None
        out.append(o)
    s["out"] = out
    if case["graph"]:
        # one pass ahead of the capture, on a side stream; the inputs that it wrote are set again
        kept = {k: s[k].clone() for k in ("x", "r") if s[k] is not None}
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _calls(s)
        torch.cuda.current_stream().wait_stream(side)
        s["captured"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["captured"]):
            s["held"] = _calls(s)
        for k, v in kept.items():
            s[k].copy_(v)
    return s


# --------------------------------------------------------------------------------------- a pass
def _call(s, k):
    name, x, w, r, ub, o = s["op"], s["x"][k], s["w"][k], s["r"], s["ub"], s["out"][k]
    if name == "add_norm_int8":
        o["q"], o["s"] = custom_ops.rms_norm_dynamic_per_token_quant(x, w, EPS, torch.int8, ub, r)
    elif name == "padded":
        p, _, rms, q, sc = custom_ops.fused_add_rms_norm_dynamic_per_token_quant_padding_output(
            x, r, w, _pad_size(s["hidden"]), EPS)
        # the bytes behind the scale are not written
        o.update(packed=p.view(torch.int8)[:, :s["hidden"] + 4], rms=rms, q=q, s=sc)
    elif name == "norm_quant":
        torch.ops._C.rms_norm_dynamic_per_token_quant(o["q"], x, w, o["s"], EPS, ub, r)
    elif name == "block_quant":
        torch.ops._C.rms_norm_per_block_quant(o["q"], x, w, o["s"], EPS, None, r, GROUP,
                                              s["transposed"])
    elif name == "fused_add_norm":
        torch.ops._C.fused_add_rms_norm(x, r, w, EPS)
        o["out"] = x
    elif name == "smooth":
        op.rms_norm_dynamic_per_token_quant(o["q"], x, w, s["sm"][k], o["s"], EPS,
                                            o["after_res"], o["after_norm"], r)
    elif name == "scale_quant":
        o["q"], o["s"] = op.scale_dynamic_quant(x, s["sm"][k], torch.int8)
    elif name in ("token_int8", "token_int8_azp"):
        torch.ops._C.dynamic_scaled_int8_quant(o["q"], x, o["s"], o.get("azp"))
    elif name == "token_fp8":
        torch.ops._C.dynamic_per_token_scaled_fp8_quant(o["q"], x, o["s"], ub)
    elif name == "norm":
        op.rms_norm(o["out"], x, w, EPS, o["after_res"], r, False)
    elif name == "vllm_norm":
        torch.ops._C.rms_norm(o["out"], x, w, EPS)
    elif name == "head_norm":
        op.head_rms_norm(o["out"], x, w, EPS, 0, s["heads"])
    return o


#: operators that update the residual in place
IN_PLACE = ("add_norm_int8", "norm_quant", "block_quant", "fused_add_norm", "padded")


def _calls(s):
    outs = [_call(s, k) for k in range(s["calls"])]
    if s["r"] is not None and s["op"] in IN_PLACE:
        outs.append({"residual": s["r"]})
    return outs


def run(state):
    if "captured" in state:
        state["captured"].replay()
        return state["held"]
    return _calls(state)


# ------------------------------------------------------------------------------- what it takes
def work(case):
    """Each input read once, each output written once."""
    T, H, e = case["tokens"], case["hidden"], DTYPES[case["dtype"]].itemsize
    heads = case.get("heads", 1)
    n, name, res = T * H * heads, case["op"], 1 if case["residual"] else 0
    data = n * e  # x
    if name in ("token_int8", "token_fp8", "scale_quant", "token_int8_azp"):
        data += n + 4 * T
    elif name in ("add_norm_int8", "norm_quant"):
        data += 2 * res * n * e + n + 4 * T
    elif name == "block_quant":
        data += 2 * res * n * e + n + 4 * (n // GROUP)
    elif name == "padded":
        data += 3 * n * e + 2 * n + 8 * T
    elif name == "fused_add_norm":
        data += 3 * n * e
    elif name == "smooth":
        data += (2 + res) * n * e + n + 4 * T
    elif name == "norm":
        data += (1 + 2 * res) * n * e
    else:
        data += n * e
    if name not in ("token_int8", "token_fp8", "token_int8_azp", "scale_quant"):
        data += H * heads * e
    if name in ("smooth", "scale_quant"):
        data += 4 * H
    if name == "token_int8_azp":
        data += 4 * T
    # squares and their sum, normalisation, weight, absmax, scaling
    return {"bytes": case["calls"] * data, "flops": case["calls"] * 8 * n}


def tolerance(case):
    """Four times what the same operators in torch with their row sums in fp32 differ by (measured
    over the listed cases and fp16 / fp32 ones)."""
    if case["quant"] == "fp8":
        # ties of codes: rel 0.0025, and one code's step is an eighth of its value
        return {"rel": 1e-2, "max": 0.45}
    if case["dtype"] == "fp32":
        # scales and outputs: rel 9e-8, largest 3.5e-7 (int8 codes: 2e-7 of them)
        return {"rel": 4e-7, "max": 2e-6, "differ": 1e-4}
    # 16-bit outputs: rel 1.7e-5, largest one bf16 step (0.008); int8 codes: 4e-7 of them differ,
    # but a single one of a small call is more than 1e-6
    return {"rel": 1e-4, "max": 0.032, "differ": 1e-4}


# --------------------------------------------------------------------------------- in 64 bits
def exact(case, seed):
    i = _inputs(case, seed)
    name, r = case["op"], None if i["r"] is None else i["r"].double()
    outs = []
    for k in range(case["calls"]):
        a, o = i["x"][k].double(), {}
        if r is not None:
            a += r
            if name in IN_PLACE:
                r = a
            elif name in ("smooth", "norm"):
                o["after_res"] = a.clone()
        elif name == "smooth":
            o["after_res"] = a.clone()
        if name in ("token_int8", "token_int8_azp", "token_fp8"):
            y = a
        elif name == "scale_quant":
            y = a * i["sm"][k].double()
        else:
            rho = (a.square().mean(-1, keepdim=True) + EPS).sqrt()
            # the SmoothQuant and head norms multiply by the root, as their definition has it
            y = (a * rho if name in ("smooth", "head_norm") else a / rho) * i["w"][k].double()
            if name in ("fused_add_norm", "norm", "vllm_norm", "head_norm"):
                o["out"] = y
            elif name == "smooth":
                o["after_norm"] = y
                y = y * i["sm"][k].double()
            elif name == "padded":
                o["rms"] = y
        top = 448.0 if case["quant"] == "fp8" else 127.0
        if name == "token_int8_azp":
            o["s"] = (y.amax(-1, keepdim=True) - y.amin(-1, keepdim=True)) / 255
        elif name == "block_quant":
            s = y.abs().reshape(case["tokens"], -1, GROUP).amax(-1) / top
            o["s"] = s.t() if case["transposed"] else s
        elif "out" not in o:
            m = y.abs().amax(-1, keepdim=True)
            m = m if i["ub"] is None else torch.minimum(m, i["ub"].double())
            o["s"] = (m / top).reshape(-1) if name == "scale_quant" else m / top
        o.update({"q": None, "packed": None, "azp": None})  # whole values
        outs.append(o)
    if r is not None and name in IN_PLACE:
        outs.append({"residual": r})
    return outs
