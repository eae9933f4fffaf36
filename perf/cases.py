"""Timed cases of the quantized-matmul path: the calls a quantized ONNX model
makes on one MI355X, through the prepared C-ABI calls that a session adapter
keeps per node.

A case is a dict of plain values whose "kind" names the call chain:

  mmi    MatMulInteger, batched, scalar or per-row / per-column zero points
  dyn    DynamicQuantizeLinear -> MatMulInteger (dynamically quantized layer)
  qlm    QLinearMatMul with host-resident scalars (statically quantized layer)
  int4   DequantizeLinear(4 bit, blocked) -> MatMul, fused, fp16
  fp8    DequantizeLinear(fp8e4m3fn, per column) -> Cast -> MatMul, fused, bf16
  gguf   DequantizePacked(gguf:*) -> Transpose -> MatMul, fused, fp16
  moe    DequantizeLinear(fp8e4m3fn experts) -> Cast -> GroupedMatMul, fused
  qconv  QLinearConv with per-channel weight scales and bias

``listed()`` names the cases, ``draw(rng)`` draws one more of the same
ranges, ``prepare`` / ``run`` make and run one, ``work`` gives the bytes and
operations it cannot do without, ``tolerance`` what another correct
implementation may differ by and ``exact`` the result in 64 bits from plain
torch.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# values per block, bytes per block
GGUF = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}


def _package():
    if "onnx_light_amd" not in sys.modules:
        path = os.path.join(ROOT, "onnx-light_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location("onnx_light_amd", path,
                                                      submodule_search_locations=[os.path.dirname(path)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["onnx_light_amd"] = mod
        spec.loader.exec_module(mod)
        mod.init(0)
    return sys.modules["onnx_light_amd"]


def listed():
    return [
        # the smallest call: one 64 x 128 product, where the launch is the cost
        {"name": "mmi_small", "kind": "mmi", "batch": 1, "M": 64, "K": 256, "N": 128, "a": "u8", "zp": "scalar"},
        # attention scores of 32 heads: small K, bound by the int32 output
        {"name": "mmi_attention", "kind": "mmi", "batch": 32, "M": 512, "K": 64, "N": 512, "a": "s8", "zp": "axis"},
        # a dynamically quantized classifier layer with sizes that divide by nothing
        {"name": "dyn_ragged", "kind": "dyn", "M": 335, "K": 1001, "N": 3001, "zp": "none"},
        # a statically quantized layer, 8 sequences decoding one token each
        {"name": "qlm_decode", "kind": "qlm", "M": 8, "K": 4096, "N": 11008, "a": "u8"},
        # the same kind of layer over a 2048-token prompt
        {"name": "qlm_prefill", "kind": "qlm", "M": 2048, "K": 4096, "N": 4096, "a": "u8"},
        # weight-only int4, decode
        {"name": "int4_decode", "kind": "int4", "M": 8, "K": 4096, "N": 11008, "block": 32, "zp": False,
         "prepared": True},
        # weight-only int4 over a prompt of ordinary length
        {"name": "int4_prompt", "kind": "int4", "M": 1000, "K": 4096, "N": 11008, "block": 32, "zp": False,
         "prepared": True},
        # fp8 weights over a long prompt: the largest
        {"name": "fp8_prefill", "kind": "fp8", "M": 4096, "K": 4096, "N": 14336},
        # a GGUF checkpoint decoding one sequence
        {"name": "gguf_decode", "kind": "gguf", "format": "q4_k", "M": 1, "K": 4096, "N": 14336},
        # a GGUF checkpoint reading a short prompt
        {"name": "gguf_prompt", "kind": "gguf", "format": "q6_k", "M": 150, "K": 4096, "N": 4096},
        # mixture of experts, 32 sequences decoding: every expert is read, none has many rows
        {"name": "moe_decode", "kind": "moe", "M": 32, "G": 8, "K": 4096, "N": 14336},
        # a quantized CNN layer at batch 32
        {"name": "qconv", "kind": "qconv", "batch": 32, "C": 256, "H": 28, "W": 28, "M": 256, "kernel": 3,
         "stride": 1},
    ]


def _log(rng, lo, hi, step=1):
    """A size from lo to hi, spread over its logarithm, a multiple of step."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step
    return min(max(v, -(-lo // step) * step), hi // step * step)


def _side(rng, lo, hi, step=1):
    """A matrix side: most are multiples of 64, the others of step only."""
    return _log(rng, lo, hi, 64 if rng.random() < 0.6 else step)


def draw(rng):
    kind = rng.choice(["mmi", "dyn", "qlm", "int4", "fp8", "gguf", "moe", "qconv"])
    if kind == "mmi":
        return {"kind": kind, "batch": _log(rng, 1, 32), "M": _side(rng, 16, 512), "K": _side(rng, 64, 256),
                "N": _side(rng, 64, 512), "a": rng.choice(["u8", "s8"]), "zp": rng.choice(["scalar", "axis"])}
    if kind == "dyn":
        return {"kind": kind, "M": _log(rng, 1, 2048), "K": _side(rng, 256, 4096), "N": _side(rng, 128, 11008),
                "zp": rng.choice(["none", "axis"])}
    if kind == "qlm":
        return {"kind": kind, "M": _log(rng, 1, 2048), "K": _side(rng, 512, 4096), "N": _side(rng, 512, 11008),
                "a": rng.choice(["u8", "s8"])}
    if kind == "int4":
        block = rng.choice([32, 128])
        return {"kind": kind, "M": _log(rng, 1, 2048), "K": _log(rng, 512, 4096, 128),
                "N": _side(rng, 512, 11008, 2), "block": block, "zp": rng.random() < 0.4,
                "prepared": rng.random() < 0.7}
    if kind == "fp8":
        return {"kind": kind, "M": _log(rng, 1, 4096), "K": _side(rng, 512, 4096), "N": _side(rng, 512, 14336)}
    if kind == "gguf":
        fmt = rng.choice(sorted(GGUF))
        return {"kind": kind, "format": fmt, "M": _log(rng, 1, 2048), "K": _log(rng, 512, 4096, 256),
                "N": _side(rng, 512, 14336)}
    if kind == "moe":
        return {"kind": kind, "M": _log(rng, 1, 1024), "G": rng.choice([4, 8, 16]), "K": _side(rng, 512, 4096, 32),
                "N": _side(rng, 512, 4096, 16)}
    side = rng.randint(7, 56)
    c = rng.choice([64, 128, 256])
    return {"kind": kind, "batch": _log(rng, 1, 32), "C": c, "H": side, "W": side, "M": rng.choice([64, 96, 128, 256]),
            "kernel": rng.choice([1, 3]), "stride": rng.choice([1, 1, 2])}


# ---- inputs -----------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _ints(g, lo, hi, shape, dtype):
    return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int32).to(dtype)


def _bytes(g, kind, shape):
    return _ints(g, 0, 256, shape, torch.uint8) if kind == "u8" else _ints(g, -128, 128, shape, torch.int8)


def _uniform(g, lo, hi, shape):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _conv_out(case):
    pad = case["kernel"] // 2
    return ((case["H"] + 2 * pad - case["kernel"]) // case["stride"] + 1,
            (case["W"] + 2 * pad - case["kernel"]) // case["stride"] + 1)


def _gguf_blocks(g, fmt, blocks):
    """Random codes with the scales of weights of moderate size."""
    raw = _ints(g, 0, 256, (blocks, GGUF[fmt][1]), torch.uint8)
    lo, hi = {"q4_0": (0.002, 0.02), "q8_0": (0.0001, 0.001), "q4_k": (0.00005, 0.0005), "q6_k": (0.00001, 0.0001)}[fmt]

    def put(at, lo, hi):
        d = _uniform(g, lo, hi, (blocks,)).to(torch.float16).view(torch.uint8).view(blocks, 2)
        raw[:, at:at + 2] = d

    put(208 if fmt == "q6_k" else 0, lo, hi)
    if fmt == "q4_k":
        put(2, lo * 7, hi * 7)
    return raw.reshape(-1)


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g = _gen(seed)
    kind, M = case["kind"], case["M"]
    if kind == "qconv":
        n, c, k = case["batch"], case["C"], case["kernel"]
        s = 1.0 / (74 * 74 * math.sqrt(c * k * k))
        return {"x": _bytes(g, "u8", (n, c, case["H"], case["W"])), "w": _bytes(g, "s8", (M, c, k, k)),
                "w_scale": _uniform(g, 20 * s, 60 * s, (M,)), "bias": _ints(g, -30000, 30000, (M,), torch.int32)}
    K, N = case["K"], case["N"]
    if kind == "mmi":
        d = {"a": _bytes(g, case["a"], (case["batch"], M, K)), "b": _bytes(g, "s8", (case["batch"], K, N))}
        if case["zp"] == "axis":
            lo = 124 if case["a"] == "u8" else -4
            d["a_zp"] = _ints(g, lo, lo + 9, (M,), d["a"].dtype)
            d["b_zp"] = _ints(g, -4, 5, (N,), torch.int8)
        return d
    if kind == "dyn":
        d = {"x": torch.randn((M, K), generator=g, device="cuda") * 3 + 0.5, "b": _bytes(g, "s8", (K, N))}
        if case["zp"] == "axis":
            d["b_zp"] = _ints(g, -4, 5, (N,), torch.int8)
        return d
    if kind == "qlm":
        return {"a": _bytes(g, case["a"], (M, K)), "b": _bytes(g, "s8", (K, N))}
    if kind == "int4":
        groups = K // case["block"]
        d = {"a": torch.randn((M, K), generator=g, device="cuda").to(torch.float16),
             "w": _ints(g, 0, 256, (K * N // 2,), torch.uint8),
             "scale": _uniform(g, 0.002, 0.02, (groups, N)).to(torch.float16)}
        if case["zp"]:
            d["zp"] = _ints(g, 0, 256, (groups * N // 2,), torch.uint8)
        return d
    if kind == "fp8":
        return {"a": torch.randn((M, K), generator=g, device="cuda").to(torch.bfloat16),
                "w": torch.randn((K, N), generator=g, device="cuda").to(torch.float8_e4m3fn),
                "scale": _uniform(g, 0.005, 0.05, (N,))}
    if kind == "gguf":
        return {"a": torch.randn((M, K), generator=g, device="cuda").to(torch.float16),
                "w": _gguf_blocks(g, case["format"], N * (K // GGUF[case["format"]][0]))}
    G = case["G"]
    return {"a": (torch.randn((M, K), generator=g, device="cuda") * 0.5).to(torch.bfloat16),
            "w": torch.randn((G, K, N), generator=g, device="cuda").to(torch.float8_e4m3fn),
            "scale": _uniform(g, 0.002, 0.022, (G, 1, N)),
            # top-2 routing: two distinct experts per token
            "index": torch.rand((M, G), generator=g, device="cuda").argsort(dim=1)[:, :2].contiguous()}


# host-resident scalars of the statically quantized layers
def _qlm_scalars(case):
    u8 = case["a"] == "u8"
    return {"a_scale": np.array(0.02, np.float32), "a_zp": np.array(128 if u8 else 3, np.uint8 if u8 else np.int8),
            "b_scale": np.array(0.005, np.float32), "b_zp": np.array(0, np.int8),
            "y_scale": np.array(0.02 * 0.005 * 74 * 74 * math.sqrt(case["K"]) / 40, np.float32),
            "y_zp": np.array(128 if u8 else 0, np.uint8 if u8 else np.int8)}


CONV = {"x_scale": np.array(0.02, np.float32), "x_zp": np.array(128, np.uint8), "w_zp": np.array(0, np.int8),
        "y_scale": np.array(0.02, np.float32), "y_zp": np.array(120, np.uint8)}


# ---- one pass ---------------------------------------------------------------

def prepare(case, seed):
    """The inputs, the prepared calls of the chain and its output buffers."""
    ol = _package()
    d = _inputs(case, seed)
    kind, M = case["kind"], case["M"]
    new = lambda shape, dtype: torch.empty(shape, dtype=dtype, device="cuda")  # noqa: E731
    if kind == "qconv":
        y = new((case["batch"], M) + _conv_out(case), torch.uint8)
        attrs = ol.conv_attrs(pads=[case["kernel"] // 2] * 4, strides=[case["stride"]] * 2)
        descs = [ol.describe(t) for t in (d["x"], CONV["x_scale"], CONV["x_zp"], d["w"], d["w_scale"], CONV["w_zp"],
                                          CONV["y_scale"], CONV["y_zp"], d["bias"])]
        call = ol.Prepared("onnxl_amd_qlinear_conv", descs + [ctypes.byref(attrs), ol.describe(y)],
                           (attrs, d, y), ol._stream_of(y))
        return {"calls": [call], "out": y}
    K, N = case["K"], case["N"]
    if kind == "mmi":
        y = new((case["batch"], M, N), torch.int32)
        za, zb = d.get("a_zp"), d.get("b_zp")
        if case["zp"] == "scalar":
            za = np.array(128, np.uint8) if case["a"] == "u8" else np.array(3, np.int8)
            zb = np.array(0, np.int8)
        return {"calls": [ol.prepare("matmul_integer", d["a"], d["b"], za, zb, y)], "out": y}
    if kind == "dyn":
        xq, s, z = new((M, K), torch.uint8), new((), torch.float32), new((), torch.uint8)
        y = new((M, N), torch.int32)
        return {"calls": [ol.prepare("dynamic_quantize_linear", d["x"], xq, s, z),
                          ol.prepare("matmul_integer", xq, d["b"], z, d.get("b_zp"), y)], "out": (xq, s, z, y)}
    if kind == "qlm":
        q = _qlm_scalars(case)
        y = new((M, N), torch.uint8 if case["a"] == "u8" else torch.int8)
        return {"calls": [ol.prepare("qlinear_matmul", d["a"], q["a_scale"], q["a_zp"], d["b"], q["b_scale"],
                                     q["b_zp"], q["y_scale"], q["y_zp"], y)], "out": y}
    if kind == "int4":
        y = new((M, N), torch.float16)
        code = ol.UINT4 if case["zp"] else ol.INT4
        descs = {3: ol.describe(d["zp"], code, tuple(d["scale"].shape))} if case["zp"] else {}
        w = d["w"]
        if case["prepared"]:
            w = ol.prepare_weight(w, code, (K, N))
        else:
            descs[1] = ol.describe(w, code, (K, N))
        return {"calls": [ol.prepare("dequantize_linear_matmul", d["a"], w, d["scale"], d.get("zp"), 0, 0, y,
                                     descs=descs)], "out": y}
    if kind == "fp8":
        y = new((M, N), torch.bfloat16)
        return {"calls": [ol.prepare("dequantize_linear_matmul", d["a"], d["w"], d["scale"], None, 1, ol.BFLOAT16,
                                     y)], "out": y}
    if kind == "gguf":
        y = new((M, N), torch.float16)
        dims = (ctypes.c_int64 * ol.MAX_RANK)(N, K)
        call = ol.Prepared("onnxl_amd_dequantize_packed_matmul",
                           [ol.describe(d["a"]), ol.describe(d["w"]), ("gguf:" + case["format"]).encode(), dims, 2,
                            ol.describe(y)], (d, y, dims), ol._stream_of(y))
        return {"calls": [call], "out": y}
    y = new((M, 2, N), torch.bfloat16)
    return {"calls": [ol.prepare("dequantize_linear_grouped_matmul", d["a"], d["w"], d["scale"], None, 1,
                                 ol.BFLOAT16, d["index"], None, 0, y)], "out": y}


def run(state):
    for call in state["calls"]:
        call()
    return state["out"]


def work(case):
    """Each input read once, each output written once; 2 operations a multiply-add."""
    kind, M = case["kind"], case["M"]
    if kind == "qconv":
        n, c, k = case["batch"], case["C"], case["kernel"]
        oh, ow = _conv_out(case)
        return {"bytes": n * c * case["H"] * case["W"] + M * c * k * k + 8 * M + n * M * oh * ow,
                "flops": 2 * n * M * oh * ow * c * k * k}
    K, N = case["K"], case["N"]
    flops = 2 * M * K * N
    if kind == "mmi":
        return {"bytes": case["batch"] * (M * K + K * N + 4 * M * N), "flops": case["batch"] * flops}
    if kind == "dyn":  # the int8 activation is an output too
        return {"bytes": 4 * M * K + M * K + K * N + 4 * M * N + 5, "flops": flops}
    if kind == "qlm":
        return {"bytes": M * K + K * N + M * N, "flops": flops}
    if kind == "int4":
        groups = K // case["block"]
        return {"bytes": 2 * M * K + K * N // 2 + groups * N * 2 + (groups * N // 2 if case["zp"] else 0) + 2 * M * N,
                "flops": flops}
    if kind == "fp8":
        return {"bytes": 2 * M * K + K * N + 4 * N + 2 * M * N, "flops": flops}
    if kind == "gguf":
        per, size = GGUF[case["format"]]
        return {"bytes": 2 * M * K + N * K // per * size + 2 * M * N, "flops": flops}
    experts = case["G"] * (1 - (1 - 2 / case["G"]) ** M)  # expected number that any token chose
    return {"bytes": int(2 * M * K + experts * (K * N + 4 * N) + 16 * M + 4 * M * N), "flops": 2 * flops}


def tolerance(case):
    """Integer results are the operators' own arithmetic, to the bit; the
    16-bit results differ by the rounding of weights and of the output."""
    kind = case["kind"]
    if kind in ("int4", "gguf"):
        return {"rel": 1.2e-3, "max": 1.2e-2}
    if kind in ("fp8", "moe"):
        return {"rel": 1e-2, "max": 5e-2}
    return "exact"


# ---- 64-bit results -----------------------------------------------------------

def _nibbles(packed, n):
    p = packed.to(torch.int32)
    return torch.stack((p & 15, p >> 4), dim=1).reshape(-1)[:n]


def _f16(raw, at):
    return raw[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)


def _gguf_values(fmt, raw):
    """The blocks' values in float64, one row a block."""
    r = raw.to(torch.int32)
    n = raw.shape[0]
    if fmt == "q4_0":
        q = r[:, 2:]
        return torch.cat((q & 15, q >> 4), dim=1).sub(8) * _f16(raw, 0)
    if fmt == "q8_0":
        return raw[:, 2:].contiguous().view(torch.int8).to(torch.float64) * _f16(raw, 0)
    if fmt == "q4_k":
        s = r[:, 4:16]
        low, high = s[:, 8:] & 15, s[:, 8:] >> 4
        sc = torch.cat((s[:, :4] & 63, low | (s[:, :4] >> 6) << 4), dim=1)
        mn = torch.cat((s[:, 4:8] & 63, high | (s[:, 4:8] >> 6) << 4), dim=1)
        q = r[:, 16:].view(n, 4, 32)
        q = torch.stack((q & 15, q >> 4), dim=2).view(n, 8, 32)
        v = q * (_f16(raw, 0) * sc).unsqueeze(2) - (_f16(raw, 2) * mn).unsqueeze(2)
        return v.reshape(n, 256)
    ql, qh = r[:, :128].view(n, 2, 64), r[:, 128:192].view(n, 2, 32)
    q = torch.stack((ql[:, :, :32] & 15 | (qh & 3) << 4, ql[:, :, 32:] & 15 | (qh >> 2 & 3) << 4,
                     ql[:, :, :32] >> 4 | (qh >> 4 & 3) << 4, ql[:, :, 32:] >> 4 | (qh >> 6 & 3) << 4), dim=2)
    sc = raw[:, 192:208].contiguous().view(torch.int8).to(torch.float64) * _f16(raw, 208)
    return (q.reshape(n, 16, 16) - 32).mul(sc.unsqueeze(2)).reshape(n, 256)


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    f = lambda t: t.to(torch.float64)  # noqa: E731
    if kind == "qconv":
        x, w, k = f(d["x"]) - 128, f(d["w"]), case["kernel"]
        oh, ow = _conv_out(case)
        cs = (torch.tensor(float(CONV["x_scale"])) * d["w_scale"].cpu() / float(CONV["y_scale"])).cuda()
        y = torch.empty((case["batch"], case["M"], oh, ow), dtype=torch.uint8, device="cuda")
        for n in range(case["batch"]):
            col = torch.nn.functional.unfold(x[n:n + 1], k, padding=k // 2, stride=case["stride"])[0]
            acc = w.reshape(case["M"], -1) @ col + f(d["bias"]).unsqueeze(1)
            v = torch.round(acc.to(torch.float32) * cs.unsqueeze(1)) + float(CONV["y_zp"])
            y[n] = v.clamp(0, 255).to(torch.uint8).view(case["M"], oh, ow)
        return y
    if kind == "mmi":
        za = f(d["a_zp"]).unsqueeze(1) if case["zp"] == "axis" else (128 if case["a"] == "u8" else 3)
        zb = f(d["b_zp"]) if case["zp"] == "axis" else 0
        return torch.stack([((f(a) - za) @ (f(b) - zb)).to(torch.int32) for a, b in zip(d["a"], d["b"])])
    if kind == "dyn":  # the scale; the integers follow the operators' own fp32 rounding
        lo, hi = min(float(d["x"].min()), 0.0), max(float(d["x"].max()), 0.0)
        return (None, torch.tensor((hi - lo) / 255, dtype=torch.float64), None, None)
    if kind == "qlm":
        q = _qlm_scalars(case)
        acc = (f(d["a"]) - int(q["a_zp"])) @ f(d["b"])
        cs = np.float32(np.float32(q["a_scale"] * q["b_scale"]) / q["y_scale"])
        v = torch.round(acc.to(torch.float32) * float(cs)) + int(q["y_zp"])
        lo, dt = (0, torch.uint8) if case["a"] == "u8" else (-128, torch.int8)
        return v.clamp(lo, lo + 255).to(dt)
    K, N = case["K"], case["N"]
    if kind == "int4":
        q = _nibbles(d["w"], K * N).view(K, N)
        groups = K // case["block"]
        if case["zp"]:
            q = q - _nibbles(d["zp"], groups * N).view(groups, N).repeat_interleave(case["block"], 0)
        else:
            q = torch.where(q > 7, q - 16, q)
        return f(d["a"]) @ (f(q) * f(d["scale"]).repeat_interleave(case["block"], 0))
    if kind == "fp8":
        return f(d["a"]) @ (f(d["w"].to(torch.float32)) * f(d["scale"]))
    if kind == "gguf":
        per, size = GGUF[case["format"]]
        w = _gguf_values(case["format"], d["w"].view(-1, size)).reshape(N, K)
        return f(d["a"]) @ w.t().contiguous()
    y = torch.empty((case["M"], 2, N), dtype=torch.float64, device="cuda")
    for e in range(case["G"]):
        m, s = torch.nonzero(d["index"] == e, as_tuple=True)
        y[m, s] = f(d["a"][m]) @ (f(d["w"][e].to(torch.float32)) * f(d["scale"][e]))
    return y
