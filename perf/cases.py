"""The work a user of this framework has it do, as cases that can be timed: each one a pass through the public entry
points (the Tripy-compatible front end `tp`, and the package's own functions over the C ABI) on operands that such a
program has in GPU memory already.

A case is a dict: "op" names the path, the other keys are its sizes, types and options.

    linear       tp.Linear, forward: quantized ("int8" with an input scale, "int4" weights only, "float8" with an input
                 scale) or plain ("none"); x is `lead` + [k], the weight [n, k], with a bias
    w4a16        block-scaled int4 weights times f16 activations [m, k]
    w8a8         per-token int8 quantization of f16 activations, then the int8 GEMM with both scales in its epilogue
    dynamic      amax, scale, quantize and (optionally) dequantize of one tensor [rows, cols] with its own scale
    static       tp.quantize, then tp.dequantize, with constant scales per tensor, per channel or per int4 block
    layernorm    tp.layernorm over the last axis
    softmax      tp.softmax over the last axis
    nvfp4        tensor amax, then block quantization to f4 with f8 block scales, then its inverse
"""
import importlib
import math

import torch

import __graft_entry__ as entry

pkg = entry.load_package()
tp = importlib.import_module(pkg.__name__ + ".tp")

_BYTES = {"float32": 4, "float16": 2, "bfloat16": 2}
_QMAX = {"int8": 127.0, "float8": 448.0, "int4": 7.0}
_CODE_BYTES = {"int8": 1.0, "float8": 1.0, "int4": 1.0}   # tp keeps one int4 code per byte

# Most work a drawn case may hold: what the largest listed ones do.
_MOST_FLOPS = 2.0 * 4096 * 4096 * 11008
_MOST_FLOPS_F32 = _MOST_FLOPS / 16                        # f32 matrix instructions run at a sixteenth of the f16 rate
_MOST_BYTES = 5.0 * 16384 * 8192


def listed():
    return [
        # One token through an attention projection of a W8A8 model: the smallest call, launches and host work count.
        dict(name="linear_int8_decode", op="linear", quant="int8", dtype="float16", batch=1, tokens=1, k=4096, n=4096),
        # The gate or up projection of a 7B-class MLP with int4 weights in blocks of 128: a decode step of a batch of 16,
        # a small prefill, a large one.
        dict(name="w4a16_decode", op="w4a16", m=16, k=4096, n=11008, block=128),
        dict(name="w4a16_short_prefill", op="w4a16", m=256, k=4096, n=11008, block=128),
        dict(name="w4a16_prefill", op="w4a16", m=4096, k=4096, n=11008, block=128),
        # The same projection as W8A8 with per-token scales, from f16 activations to f16 results.
        dict(name="w8a8_prefill", op="w8a8", m=2048, k=4096, n=11008),
        # A float8 Linear of a bf16 model on three sequences of an odd length.
        dict(name="linear_float8_prefill", op="linear", quant="float8", dtype="bfloat16", batch=3, tokens=333, k=4096, n=11008),
        # Calibration-free int8 quantization of one layer's f32 activations, and its inverse.
        dict(name="dynamic_int8", op="dynamic", dtype="float32", code="int8", rows=1024, cols=4096, dequantize=True),
        # Dynamic float8 quantization of a long batch's bf16 activations with outliers, and its inverse: the largest tensor.
        dict(name="dynamic_float8_large", op="dynamic", dtype="bfloat16", code="float8", rows=16384, cols=8192, dequantize=True),
        # Block-wise int4 fake quantization of a weight matrix through the front end.
        dict(name="static_int4_block", op="static", dtype="bfloat16", code="int4", mode="block", rows=4096, cols=11008),
        # The normalisation between two layers, 8192 tokens.
        dict(name="layernorm_bf16", op="layernorm", dtype="bfloat16", rows=8192, d=4096),
        # Attention scores of eight sequences and twelve heads, 500 queries by 1500 keys: rows that are no power of two.
        dict(name="softmax_scores", op="softmax", dtype="float16", batch=8, heads=12, rows=500, d=1500),
        # NVFP4 of a prefill's activations and its inverse.
        dict(name="nvfp4", op="nvfp4", dtype="bfloat16", rows=4096, cols=8192, axis=-1),
    ]


# ---- more cases of the same ranges ---------------------------------------------------------------
def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _features(rng, lo, hi, step):
    """A feature count: a whole number of `step`, or (one in six) any number."""
    v = _log(rng, lo, hi)
    return v if step > 1 and rng.random() < 1 / 6 else max(step, v // step * step)


def _multiple(rng, lo, hi, step):
    return max(step, _log(rng, lo, hi) // step * step)


def _tokens(m, most):
    return max(1, min(m, int(most)))


def draw(rng):
    op = rng.choice(["linear", "linear", "linear", "w4a16", "w4a16", "w8a8", "w8a8", "dynamic", "dynamic", "static", "layernorm", "softmax", "nvfp4"])
    if op == "linear":
        quant = rng.choice(["int8", "int4", "float8", "none"])
        dtype = {"int8": "float16", "int4": "float16", "float8": rng.choice(["bfloat16", "float16"]),
                 "none": rng.choice(["float16", "bfloat16", "float32"])}[quant]
        k, n = _features(rng, 256, 12288, 64), _features(rng, 256, 16384, 64)
        m = _tokens(_log(rng, 1, 4096), (_MOST_FLOPS_F32 if dtype == "float32" else _MOST_FLOPS) / (2.0 * k * n))
        batch = rng.choice([1, 1, 2, 3, 4])
        return dict(op=op, quant=quant, dtype=dtype, batch=batch, tokens=max(1, m // batch), k=k, n=n)
    if op == "w4a16":
        block = rng.choice([64, 128, 128, 128, 256])
        k, n = _multiple(rng, 512, 14336, max(block, 128)), _features(rng, 256, 16384, 64)
        return dict(op=op, m=_tokens(_log(rng, 1, 4096), _MOST_FLOPS / (2.0 * k * n)), k=k, n=n, block=block)
    if op == "w8a8":
        k, n = _multiple(rng, 512, 14336, 128), _features(rng, 256, 16384, 64)
        return dict(op=op, m=_tokens(_log(rng, 1, 4096), _MOST_FLOPS / (2.0 * k * n)), k=k, n=n)
    dtype = rng.choice(["float32", "float16", "bfloat16"])
    if op == "nvfp4":
        rows, cols = _multiple(rng, 16, 16384, 16), _multiple(rng, 64, 16384, 16)
        axis = rng.choice([-1, -1, -2])
        rows = max(16, min(rows, int(_MOST_BYTES / (2.0 * cols * (_BYTES[dtype] + 1))) // 16 * 16))
        return dict(op=op, dtype=dtype, rows=rows, cols=cols, axis=axis)
    if op == "softmax":
        d = _log(rng, 16, 65536)
        rows = max(1, min(_log(rng, 1, 65536), int(_MOST_BYTES / (2.0 * d * _BYTES[dtype]))))
        heads = rng.choice([1, 4, 12])
        return dict(op=op, dtype=dtype, batch=1, heads=heads, rows=max(1, rows // heads), d=d)
    if op == "layernorm":
        d = _features(rng, 64, 16384, 64)
        return dict(op=op, dtype=dtype, rows=max(1, min(_log(rng, 1, 32768), int(_MOST_BYTES / (2.0 * d * _BYTES[dtype])))), d=d)
    cols = _features(rng, 64, 16384, 64)
    rows = max(1, min(_log(rng, 1, 32768), int(_MOST_BYTES / (2.0 * cols * (_BYTES[dtype] + 1)))))
    if op == "dynamic":
        return dict(op=op, dtype=dtype, code=rng.choice(["int8", "float8"]), rows=rows, cols=cols, dequantize=rng.random() < 0.6)
    mode = rng.choice(["tensor", "channel0", "channel1", "block"])
    code = "int4" if mode == "block" else rng.choice(["int8", "int8", "float8", "int4"])
    if mode == "block":
        rows = max(128, rows // 128 * 128)
        cols = max(1, min(cols, int(_MOST_BYTES / (2.0 * rows * (_BYTES[dtype] + 1)))))
    return dict(op=op, dtype=dtype, code=code, mode=mode, rows=rows, cols=cols)


# ---- what a program has in hand before the call --------------------------------------------------
def _normal(gen, shape, dtype, std=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * std).to(getattr(torch, dtype))


def _uniform(gen, shape, lo, hi):
    return torch.rand(shape, generator=gen, device="cuda") * (hi - lo) + lo


def _prepare_linear(c, gen):
    k, n, dtype = c["k"], c["n"], getattr(tp, c["dtype"])
    quant = None if c["quant"] == "none" else getattr(tp, c["quant"])
    x = _normal(gen, (c["batch"], c["tokens"], k), c["dtype"])
    w = _normal(gen, (n, k), c["dtype"], 1.0 / math.sqrt(k))
    state = {"weight": tp.Tensor(w), "bias": tp.Tensor(_normal(gen, (n,), c["dtype"], 0.1))}
    lin = tp.Linear(k, n, dtype=dtype, quant_dtype=quant, weight_quant_dim=None if quant is None else 0)
    if quant is not None:
        # scales are calibration constants in host memory, in the module's type
        state["weight_scale"] = tp.Tensor((w.float().abs().amax(dim=1) / _QMAX[c["quant"]]).to(w.dtype).cpu())
        if c["quant"] != "int4":
            state["input_scale"] = tp.Tensor((torch.tensor(5.0) / _QMAX[c["quant"]]).to(w.dtype))
    lin.load_state_dict(state)
    return {"linear": lin, "x": tp.Tensor(x)}


def _prepare_static(c, gen):
    rows, cols, qmax = c["rows"], c["cols"], _QMAX[c["code"]]
    x = _normal(gen, (rows, cols), c["dtype"], 0.02)
    shape = {"tensor": (), "channel0": (rows,), "channel1": (cols,), "block": (rows // 128, cols)}[c["mode"]]
    scale = _uniform(gen, shape, 0.05, 0.1) / qmax
    return {"x": tp.Tensor(x), "scale": tp.Tensor(scale.to(x.dtype).cpu()), "code": getattr(tp, c["code"]), "dtype": getattr(tp, c["dtype"]),
            "dim": {"channel0": 0, "channel1": 1}.get(c["mode"])}


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    op = c["op"]
    s = {}
    if op == "linear":
        s = _prepare_linear(c, gen)
    elif op == "w4a16":
        m, k, n = c["m"], c["k"], c["n"]
        packed = torch.randint(0, 256, ((k * n + 1) // 2,), generator=gen, device="cuda", dtype=torch.uint8)
        s = {"a": _normal(gen, (m, k), "float16"), "w": pkg.gemm_w4a16_prepack(packed, k, n),
             "scale": _uniform(gen, (k // c["block"], n), 0.005, 0.02).half()}
    elif op == "w8a8":
        k, n = c["k"], c["n"]
        w = torch.clamp(torch.round(_normal(gen, (k, n), "float32", 40.0)), -128, 127).to(torch.int8)
        s = {"x": _normal(gen, (c["m"], k), "float16"), "w": pkg.gemm_w8a8_prepack_fragments(w),
             "w_scale": _uniform(gen, (n,), 1e-4, 4e-4)}
    elif op == "dynamic":
        x = _normal(gen, (c["rows"], c["cols"]), "float32", math.sqrt(2.0))
        if c["code"] == "float8":                         # activations with outliers: one in a thousand, fifty times as large
            x = torch.where(torch.rand(x.shape, generator=gen, device="cuda") < 0.001, x * 50.0, x)
        s = {"x": x.to(getattr(torch, c["dtype"])), "code": {"int8": pkg.I8, "float8": pkg.F8E4M3FN}[c["code"]]}
    elif op == "static":
        s = _prepare_static(c, gen)
    elif op == "layernorm":
        d = c["d"]
        s = {"x": tp.Tensor(_normal(gen, (c["rows"], d), c["dtype"])),
             "gamma": tp.Tensor(_uniform(gen, (d,), 0.5, 1.5).to(getattr(torch, c["dtype"]))),
             "beta": tp.Tensor(_normal(gen, (d,), c["dtype"], 0.1))}
    elif op == "softmax":
        s = {"x": tp.Tensor(_normal(gen, (c["batch"], c["heads"], c["rows"], c["d"]), c["dtype"], 2.0))}
    elif op == "nvfp4":
        s = {"x": _normal(gen, (c["rows"], c["cols"]), c["dtype"])}
    else:
        raise ValueError("unknown op %r" % (op,))
    s["case"] = dict(c)
    return s


# ---- one pass ------------------------------------------------------------------------------------
def run(state):
    c = state["case"]
    op = c["op"]
    if op == "linear":
        return state["linear"](state["x"]).torch()
    if op == "w4a16":
        return pkg.gemm_w4a16(state["a"], state["scale"], c["k"], c["n"], c["block"], w_prepacked=state["w"])
    if op == "w8a8":
        q, _, scale = pkg.dynamic_quantize_rows(state["x"], pkg.I8, 127.0, want_amax=False)
        y = pkg.gemm_w8a8_fragments(q.view(c["m"], c["k"]), state["w"], scale, state["w_scale"], c["n"])
        return {"q": q, "scale": scale, "y": y}
    if op == "dynamic":
        q, y, amax, scale = pkg.dynamic_quantize_dequantize(state["x"], state["code"], _QMAX[c["code"]], dequantize=c["dequantize"])
        return {"q": q, "y": y, "amax": amax, "scale": scale}
    if op == "static":
        q = tp.quantize(state["x"], state["scale"], state["code"], state["dim"])
        y = tp.dequantize(q, state["scale"], state["dtype"], state["dim"])
        return {"q": q.torch(), "y": y.torch()}
    if op == "layernorm":
        return tp.layernorm(state["x"], state["gamma"], state["beta"], 1e-5).torch()
    if op == "softmax":
        return tp.softmax(state["x"], dim=-1).torch()
    x = state["x"]
    amax, _ = pkg.amax(x, 2688.0)
    q, scales = pkg.nvfp4_quantize(x, amax, axis=c["axis"])
    y = pkg.nvfp4_dequantize(q, scales, amax, x.dtype, x.shape, axis=c["axis"])
    return {"q": q, "scales": scales, "y": y, "amax": amax}


# ---- what a pass cannot do without, and how close another implementation comes -------------------
def work(case):
    c = case
    op = c["op"]
    flops = 0.0
    if op == "linear":
        m, k, n, b = c["batch"] * c["tokens"], c["k"], c["n"], _BYTES[c["dtype"]]
        weight = {"int8": 1.0, "float8": 1.0, "int4": 0.5, "none": b}[c["quant"]]
        scales = 0 if c["quant"] == "none" else n * b
        nbytes, flops = m * k * b + weight * k * n + scales + n * b + m * n * b, 2.0 * m * k * n
    elif op == "w4a16":
        m, k, n = c["m"], c["k"], c["n"]
        nbytes, flops = 2.0 * m * k + k * n / 2 + 2.0 * (k // c["block"]) * n + 2.0 * m * n, 2.0 * m * k * n
    elif op == "w8a8":
        m, k, n = c["m"], c["k"], c["n"]
        nbytes, flops = 3.0 * m * k + 4.0 * m + k * n + 4.0 * n + 2.0 * m * n, 2.0 * m * k * n
    elif op == "dynamic":
        e, b = c["rows"] * c["cols"], _BYTES[c["dtype"]]
        nbytes = e * (b + 1.0 + (b if c["dequantize"] else 0)) + 8
    elif op == "static":
        e, b = c["rows"] * c["cols"], _BYTES[c["dtype"]]
        nbytes = e * (2.0 * b + _CODE_BYTES[c["code"]])
        nbytes += 4.0 * {"tensor": 1, "channel0": c["rows"], "channel1": c["cols"], "block": c["rows"] // 128 * c["cols"]}[c["mode"]]
    elif op == "layernorm":
        nbytes = _BYTES[c["dtype"]] * (2.0 * c["rows"] * c["d"] + 2.0 * c["d"])
    elif op == "softmax":
        nbytes = _BYTES[c["dtype"]] * 2.0 * c["batch"] * c["heads"] * c["rows"] * c["d"]
    else:
        nbytes = c["rows"] * c["cols"] * (2.0 * _BYTES[c["dtype"]] + 0.5 + 1.0 / 16) + 4
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    """Codes, scales and dequantized values are defined bit for bit; results of float sums by the rounding of their type."""
    if case["op"] in ("dynamic", "static", "nvfp4"):
        return "exact"
    dtype = case.get("dtype", "float16")
    return {"rel": {"float32": 1e-5, "float16": 1e-3, "bfloat16": 5e-3}[dtype]}
