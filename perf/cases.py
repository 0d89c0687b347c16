"""The work that a user of this library has it do, as cases that can be timed and compared.

A case is a dict of plain values.  ``listed()`` names twelve: the operators of an ONNX
inference graph, each through the C ABI on device-resident tensors (the caller owns the
output buffers, as the ABI has it), and two whole graphs through the Python executor.
``draw(rng)`` gives further cases of the same ranges: odd and ragged sizes, both storage
orders of a Gemm's weight, every axis and code type of the quantization operators, plain,
strided, shallow and depthwise convolutions, float32 and float16.

``prepare`` makes what a program holds before the call, ``run`` makes the call, ``exact``
restates it in 64 bits with plain torch.
"""
import ctypes
import math

import numpy as np
import torch

from onnx_translator_amd.nn import DTYPE_MAP, PT, Ops, Tensor
from onnx_translator_amd.nn.Operators import CConvParams, CPoolParams

DEVICE = "cuda"
TORCH_DTYPE = {"float32": torch.float32, "float16": torch.float16, "int8": torch.int8, "uint8": torch.uint8,
               "float8_e4m3": torch.uint8, "float8_e5m2": torch.uint8}
ELEM_BYTES = {"float32": 4, "float16": 2, "int8": 1, "uint8": 1, "float8_e4m3": 1, "float8_e5m2": 1}
# largest magnitude a code type represents: scale = max |x| / this
CODE_MAX = {"int8": 127.0, "uint8": 255.0, "float8_e4m3": 448.0, "float8_e5m2": 57344.0}
BINARY = ("add", "sub", "mul", "div")


def listed():
    return [
        # A per-channel bias on a small activation: the smallest call there is, where the
        # launch and the way to it count as much as the 12.8 MB.
        {"name": "add_channel_bias", "op": "binary", "fn": "add", "n": 8, "c": 64, "h": 56, "w": 56,
         "channel": True, "dtype": "float32"},
        # Per-axis int8 quantization of a [batch, channels, features] activation and its
        # dequantization: what calibration and fake quantization run over whole activations.
        {"name": "quantize_pair_axis", "op": "qdq", "n": 32, "c": 512, "r": 1024, "axis": 1, "code": "int8"},
        # Attention-like row softmax: many short rows of an odd length.
        {"name": "softmax_short_rows", "op": "softmax", "outer": 24576, "len": 257, "inner": 1, "dtype": "float32"},
        # The 2x2 pooling between convolution stages.
        {"name": "maxpool_2x2", "op": "maxpool", "n": 32, "c": 64, "h": 112, "w": 112, "k": 2, "s": 2, "p": 0},
        # A dense layer with the weight stored [in, out] (ONNX's default, transB = 0).
        {"name": "gemm_f32_in_out", "op": "gemm", "m": 512, "n": 4096, "k": 1024, "tb": 0, "dtype": "float32"},
        # The large half-precision product, weight stored [out, in]: the most work of one call.
        {"name": "gemm_f16_large", "op": "gemm", "m": 4096, "n": 4096, "k": 4096, "tb": 1, "dtype": "float16"},
        # A weight-only-quantized layer at a small serving batch: one pass over the int8 weight.
        {"name": "woq_gemm_small_batch", "op": "woq", "m": 8, "n": 4096, "k": 4096},
        # The 3x3 convolution of a residual stage.
        {"name": "conv_3x3", "op": "conv", "n": 32, "c": 64, "h": 56, "w": 56, "m": 64, "k": 3, "s": 1,
         "depthwise": False, "dtype": "float32"},
        # A depthwise 3x3 convolution: one filter per channel, no reduction over channels.
        {"name": "conv_depthwise", "op": "conv", "n": 32, "c": 96, "h": 56, "w": 56, "m": 96, "k": 3, "s": 1,
         "depthwise": True, "dtype": "float32"},
        # The convolution of a half-precision model.
        {"name": "conv_3x3_f16", "op": "conv", "n": 32, "c": 128, "h": 28, "w": 28, "m": 128, "k": 3, "s": 1,
         "depthwise": False, "dtype": "float16"},
        # One image through the quantized residual network, default graph passes: latency.
        {"name": "graph_qdq_one_image", "op": "graph", "batch": 1, "int8": False},
        # A serving batch through the same network with its blocks on integer codes.
        {"name": "graph_int8_batch", "op": "graph", "batch": 64, "int8": True},
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _edge(rng, lo, hi):
    """As _log, rounded to a multiple of 16 half of the time (layers are wide in such steps)."""
    v = _log(rng, lo, hi)
    return v if rng.random() < 0.5 or v < 16 else v // 16 * 16


def draw(rng):
    op = rng.choice(["binary", "qdq", "softmax", "maxpool", "gemm", "gemm", "woq", "conv", "conv", "graph"])
    if op == "binary":
        n, c, hw = _log(rng, 1, 32), _log(rng, 16, 512), _log(rng, 7, 112)
        while n * c * hw * hw > 1 << 24:
            n, c = max(1, n // 2), max(8, c // 2)
        return {"op": op, "fn": rng.choice(BINARY), "n": n, "c": c, "h": hw, "w": hw,
                "channel": rng.random() < 0.6, "dtype": rng.choice(["float32", "float32", "float16"])}
    if op == "qdq":
        # activations [batch, channels, pixels or features], weights [rows, 1, columns];
        # axis 0: per output row, 1: per channel, 2: per output column, -1: one scale
        n, c, r = _log(rng, 1, 64), _log(rng, 1, 1024), _edge(rng, 9, 8192)
        while n * c * r > 1 << 24:
            n, c = max(1, n // 2), max(1, c // 2)
        return {"op": op, "n": n, "c": c, "r": r, "axis": rng.choice([-1, -1, 0, 1, 2]),
                "code": rng.choice(["int8", "uint8", "float8_e4m3", "float8_e5m2"])}
    if op == "softmax":
        length, outer = _log(rng, 10, 32000), _log(rng, 1, 32768)
        while length * outer > 1 << 23:
            outer = max(1, outer // 2)
        # over the channels of an [outer, channels, pixels] map one time in four
        inner = 1
        if rng.random() < 0.25:
            length, inner = _log(rng, 10, 512), _log(rng, 16, 4096)
            outer = max(1, min(outer, 64, (1 << 23) // (length * inner)))
        return {"op": op, "outer": outer, "len": length, "inner": inner,
                "dtype": rng.choice(["float32", "float32", "float16"])}
    if op == "maxpool":
        k, s, p = rng.choice([(2, 2, 0), (3, 2, 1), (3, 2, 0), (3, 1, 1), (5, 1, 2)])
        hw, c, n = _log(rng, 7, 128), _log(rng, 16, 512), _log(rng, 1, 32)
        while n * c * hw * hw > 1 << 25:
            n, c = max(1, n // 2), max(8, c // 2)
        return {"op": op, "n": n, "c": c, "h": hw, "w": hw, "k": k, "s": s, "p": p}
    if op == "gemm":
        dtype = rng.choice(["float32", "float16"])
        m, n, k = _log(rng, 1, 2048), _edge(rng, 64, 4096), _edge(rng, 64, 4096)
        return {"op": op, "m": m, "n": n, "k": k, "tb": rng.choice([0, 1]), "dtype": dtype}
    if op == "woq":
        return {"op": op, "m": _log(rng, 1, 256), "n": _edge(rng, 256, 8192), "k": _edge(rng, 256, 4096) // 4 * 4}
    if op == "conv":
        k, s = rng.choice([(1, 1), (3, 1), (3, 1), (3, 2), (5, 1)])
        hw, n, c = _log(rng, 7, 112), _log(rng, 1, 32), _edge(rng, 8, 512)
        depthwise = k > 1 and rng.random() < 0.3
        m = c if depthwise else _edge(rng, 8, 512)
        while n > 1 and (n * max(c, m) * hw * hw > 1 << 24 or
                         2 * n * m * (1 if depthwise else c) * k * k * hw * hw / (s * s) > 15e9):
            n //= 2
        return {"op": op, "n": n, "c": c, "h": hw, "w": hw, "m": m, "k": k, "s": s, "depthwise": depthwise,
                "dtype": rng.choice(["float32", "float32", "float16"])}
    return {"op": op, "batch": _log(rng, 1, 64), "int8": rng.choice([False, True])}


# ---------------------------------------------------------------- the library ---
_LIB = None


def _lib():
    """The operator library, with the signatures of the entry points used here."""
    global _LIB
    if _LIB is None:
        lib = Ops._get_lib()
        cf, ci = ctypes.c_float, ctypes.c_int
        lib.gemm_forward.argtypes = [PT, PT, PT, PT, cf, cf, ci, ci]
        lib.dequantize_gemm_forward.argtypes = [PT, PT, PT, PT, ci, PT, PT, cf, cf, ci, ci]
        lib.softmax_forward.argtypes = [PT, PT, ci]
        lib.max_pool_forward.argtypes = [PT, PT, ctypes.POINTER(CPoolParams)]
        lib.conv2d_forward.argtypes = [PT, PT, PT, PT, ctypes.POINTER(CConvParams)]
        _LIB = lib
    return _LIB


def _wrap(lib, t, dtype=None):
    """A library tensor over a torch tensor's memory (the caller keeps the torch tensor)."""
    shape = tuple(t.shape) or (1,)
    name = dtype or next(k for k, v in TORCH_DTYPE.items() if v == t.dtype)
    return lib.tensor_wrap_device(ctypes.c_void_p(t.data_ptr()), (ctypes.c_int * len(shape))(*shape), len(shape),
                                  DTYPE_MAP[name])


def _ints(*v):
    return (ctypes.c_int * len(v))(*v)


def _out_hw(case):
    p = case.get("p", case["k"] // 2)
    return ((case["h"] + 2 * p - case["k"]) // case["s"] + 1, (case["w"] + 2 * p - case["k"]) // case["s"] + 1, p)


# --------------------------------------------------------------------- inputs ---
def _inputs(case, seed):
    """The case's input tensors, from the seed alone."""
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))

    def normal(*shape, std=1.0, dtype="float32"):
        return (torch.randn(*shape, generator=g, device=DEVICE) * std).to(TORCH_DTYPE[dtype])

    op = case["op"]
    if op == "binary":
        dt = case["dtype"]
        a = normal(case["n"], case["c"], case["h"], case["w"], dtype=dt)
        b = normal(*((case["c"], 1, 1) if case["channel"] else a.shape), dtype=dt)
        # divisors and factors are scales: away from zero
        return (a, b.abs() + 0.5 if case["fn"] in ("mul", "div") else b)
    if op == "qdq":
        x = normal(case["n"], case["c"], case["r"], std=1.5)
        unsigned = case["code"] == "uint8"
        if case["axis"] < 0:
            span = (x.amax() - x.amin()) if unsigned else x.abs().amax()
            s = (span / CODE_MAX[case["code"]]).reshape(1)
        else:
            dims = [d for d in range(3) if d != case["axis"]]
            span = (x.amax(dims) - x.amin(dims)) if unsigned else x.abs().amax(dims)
            s = torch.clamp(span, min=0.1) / CODE_MAX[case["code"]]
        z = torch.full(s.shape, 128 if unsigned else 0, device=DEVICE, dtype=TORCH_DTYPE[case["code"]])
        return x, s.float(), z
    if op == "softmax":
        return (normal(case["outer"], case["len"], case["inner"], std=2.0, dtype=case["dtype"]),)
    if op == "maxpool":
        return (normal(case["n"], case["c"], case["h"], case["w"]).relu_(),)
    if op == "gemm":
        m, n, k, dt = case["m"], case["n"], case["k"], case["dtype"]
        w = normal(*((n, k) if case["tb"] else (k, n)), std=1 / math.sqrt(k), dtype=dt)
        return normal(m, k, dtype=dt), w, normal(n, std=0.1)
    if op == "woq":
        m, n, k = case["m"], case["n"], case["k"]
        w = normal(n, k, std=1 / math.sqrt(k))
        s = w.abs().amax(1) / 127
        q = torch.clamp(torch.round(w / s[:, None]), -127, 127).to(torch.int8)
        return normal(m, k), q, s, torch.zeros(n, dtype=torch.int8, device=DEVICE), normal(n, std=0.1)
    if op == "conv":
        cg = 1 if case["depthwise"] else case["c"]
        x = normal(case["n"], case["c"], case["h"], case["w"], dtype=case["dtype"])
        w = normal(case["m"], cg, case["k"], case["k"], std=math.sqrt(2 / (cg * case["k"] ** 2)), dtype=case["dtype"])
        return x.relu_(), w, normal(case["m"], std=0.1)
    raise ValueError(op)


def _model(case, seed):
    """The residual network with its logits as a second output, and a batch of images."""
    from onnx_translator_amd.onnx.create_model import resnet_qdq_model
    from onnx_translator_amd.onnx.proto import FLOAT, ValueInfoProto
    model = resnet_qdq_model(batch=case["batch"], seed=int(seed) % 1000003)
    model.graph.outputs.append(ValueInfoProto("logits", FLOAT, [case["batch"], 1000]))
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return model, torch.randn(case["batch"], 3, 224, 224, generator=g, device=DEVICE)


def prepare(case, seed):
    lib = _lib()
    op = case["op"]
    if op == "graph":
        from onnx_translator_amd.nn import DeviceArray
        from onnx_translator_amd.nn.ONNXImport import load_graph
        model, x = _model(case, seed)
        graph = load_graph(model, fuse=False)
        graph.fuse(int8_conv=case["int8"])
        torch.cuda.synchronize()
        held = Tensor(*x.shape, dtype="float32", data=DeviceArray(lib, x.shape, "float32", ptr=_wrap(lib, x)))
        return {"op": op, "graph": graph, "x": held, "keep": x}
    ins = _inputs(case, seed)
    st = {"op": op, "lib": lib, "keep": ins, "in": [_wrap(lib, t) for t in ins]}
    dt = TORCH_DTYPE[case.get("dtype", "float32")]
    if op in ("binary", "softmax"):
        st["out"] = [torch.empty(ins[0].shape, dtype=dt, device=DEVICE)]
        st["fn"] = case.get("fn", "")
    elif op == "qdq":
        code = case["code"]
        st["out"] = [torch.empty(ins[0].shape, dtype=TORCH_DTYPE[code], device=DEVICE), torch.empty_like(ins[0])]
        st["in"][2] = _wrap(lib, ins[2], code)
        st["code"] = _wrap(lib, st["out"][0], code)
        st["axis"] = case["axis"]
    elif op in ("maxpool", "conv"):
        oh, ow, p = _out_hw(case)
        m = case.get("m", case["c"])
        st["out"] = [torch.empty(case["n"], m, oh, ow, dtype=dt, device=DEVICE)]
        st["ints"] = [_ints(p, p, p, p), _ints(case["s"], case["s"]), _ints(1, 1), _ints(case["k"], case["k"])]
        group = case["c"] if case.get("depthwise") else 1
        st["params"] = CConvParams(*st["ints"][:3], group) if op == "conv" else CPoolParams(*st["ints"])
    elif op in ("gemm", "woq"):
        st["out"] = [torch.empty(case["m"], case["n"], dtype=dt, device=DEVICE)]
        st["tb"] = case.get("tb", 1)
    st["to"] = [_wrap(lib, t) for t in st["out"]]
    if op == "qdq":
        st["to"][0] = st["code"]
    torch.cuda.synchronize()      # the library's stream is its own: the inputs are written
    return st


# ----------------------------------------------------------------------- call ---
def run(st):
    op = st["op"]
    if op == "graph":
        probs, logits = st["graph"].forward(st["x"])
        return {"logits": logits.numpy(), "probs": probs.numpy()}
    lib, i, o = st["lib"], st["in"], st["to"]
    if op == "binary":
        getattr(lib, st["fn"] + "_forward")(i[0], i[1], o[0])
    elif op == "qdq":
        if st["axis"] < 0:
            lib.quantize_linear_forward(i[0], i[1], i[2], o[0])
            lib.dequantize_linear_forward(o[0], i[1], i[2], o[1])
        else:
            lib.quantize_linear_axis_forward(i[0], i[1], i[2], o[0], st["axis"])
            lib.dequantize_linear_axis_forward(o[0], i[1], i[2], o[1], st["axis"])
    elif op == "softmax":
        lib.softmax_forward(i[0], o[0], 1)
    elif op == "maxpool":
        lib.max_pool_forward(i[0], o[0], ctypes.byref(st["params"]))
    elif op == "conv":
        lib.conv2d_forward(i[0], i[1], i[2], o[0], ctypes.byref(st["params"]))
    elif op == "gemm":
        lib.gemm_forward(i[0], i[1], i[2], o[0], 1.0, 1.0, 0, st["tb"])
    else:
        lib.dequantize_gemm_forward(i[0], i[1], i[2], i[3], 0, i[4], o[0], 1.0, 1.0, 0, 1)
    err = lib.tensor_ops_hip_last_error()
    if err:
        raise RuntimeError(err.decode())
    return st["out"]


# ------------------------------------------------------------ work, tolerance ---
def work(case):
    op = case["op"]
    if op == "binary":
        e = case["n"] * case["c"] * case["h"] * case["w"]
        return {"bytes": ELEM_BYTES[case["dtype"]] * (2 * e + (case["c"] if case["channel"] else e)), "flops": e}
    if op == "qdq":
        e = case["n"] * case["c"] * case["r"]
        return {"bytes": 10 * e, "flops": 4 * e}       # 4 B in, 1 B out, then 1 B in, 4 B out
    if op == "softmax":
        e = case["outer"] * case["len"] * case["inner"]
        return {"bytes": 2 * e * ELEM_BYTES[case["dtype"]], "flops": 5 * e}
    if op == "maxpool":
        oh, ow, _ = _out_hw(case)
        planes = case["n"] * case["c"]
        return {"bytes": 4 * planes * (case["h"] * case["w"] + oh * ow), "flops": planes * oh * ow * case["k"] ** 2}
    if op == "gemm":
        m, n, k, b = case["m"], case["n"], case["k"], ELEM_BYTES[case["dtype"]]
        return {"bytes": b * (m * k + n * k + m * n) + 4 * n, "flops": 2 * m * n * k}
    if op == "woq":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * m * k + n * k + 9 * n + 4 * m * n, "flops": 2 * m * n * k}
    if op == "conv":
        oh, ow, _ = _out_hw(case)
        b, kg = ELEM_BYTES[case["dtype"]], (1 if case["depthwise"] else case["c"]) * case["k"] ** 2
        out = case["n"] * case["m"] * oh * ow
        return {"bytes": b * (case["n"] * case["c"] * case["h"] * case["w"] + case["m"] * kg + out) + 4 * case["m"],
                "flops": 2 * out * kg}
    per_image = 2 * (64 * 112 * 112 * 147 + 64 * 56 * 56 * 576 + 128 * 28 * 28 * (576 + 64) +
                     256 * 14 * 14 * (1152 + 128) + 512 * 7 * 7 * (2304 + 256) + 1000 * 512)
    weights = 64 * 147 * 4 + 64 * 576 + 128 * 640 + 256 * 1280 + 512 * 2560 + 4 * 1000 * 513
    return {"bytes": case["batch"] * 4 * (3 * 224 * 224 + 2000) + weights, "flops": case["batch"] * per_image}


def tolerance(case):
    op = case["op"]
    if op in ("binary", "qdq", "maxpool"):
        return "exact"                                  # bit for bit by contract
    half = case.get("dtype") == "float16"
    if op == "softmax":
        # outputs a few units in the last place apart
        return {"rel": 4e-4, "max": 4e-3} if half else {"rel": 1e-6, "max": 1e-5}
    if op in ("gemm", "woq", "conv"):
        # float32 sums in another order; a float16 result may round to the neighbouring value
        return {"rel": 4e-4, "max": 4e-3} if half else {"rel": 4e-6, "max": 1e-4}
    # another order of a convolution's sums moves a few activation codes by one step
    # (the probabilities are then 2e-4 off the 64-bit ones)
    return {"rel": 1e-3, "max": 1e-2}


# -------------------------------------------------------------------- 64 bits ---
def _conv64(x, w, b, stride, pad, group=1):
    n, c, h, wd = x.shape
    m, cg, k, _ = w.shape
    oh, ow = (h + 2 * pad - k) // stride + 1, (wd + 2 * pad - k) // stride + 1
    wg = w.double().reshape(group, m // group, cg * k * k)
    out = torch.empty(n, m, oh, ow, dtype=torch.float64, device=x.device)
    step = max(1, (1 << 28) // (c * k * k * oh * ow * 8))
    for i in range(0, n, step):
        cols = torch.nn.functional.unfold(x[i:i + step].double(), k, padding=pad, stride=stride)
        cols = cols.reshape(-1, group, cg * k * k, oh * ow)
        out[i:i + step] = torch.matmul(wg, cols).reshape(-1, m, oh, ow)
    return out if b is None else out + b.double().reshape(1, m, 1, 1)


def _graph64(case, seed):
    """The network's operators in order, in 64 bits, from the weights in the model."""
    model, x = _model(case, seed)
    w = {t.name: torch.from_numpy(np.array(t.numpy())).to(DEVICE) for t in model.graph.initializers}
    step = w["act.scale"].double()

    def weight(p):
        return w[p + ".wq"].double() * w[p + ".ws"].double().reshape(-1, 1, 1, 1)

    y = torch.relu(_conv64(x, w["stem.w"], w["stem.b"], 2, 3))
    y = torch.nn.functional.max_pool2d(y, 3, 2, 1)
    for i in range(1, 5):
        p, stride = "block%d" % i, 1 if i == 1 else 2
        act = torch.clamp(torch.round(y / step), 0, 255) * step
        main = torch.relu(_conv64(act, weight(p), w[p + ".b"], stride, 1))
        y = main + (y if i == 1 else _conv64(act, weight(p + ".proj"), None, stride, 0))
    logits = y.mean((2, 3)) @ w["fc.w"].double().t() + w["fc.b"].double()
    return {"logits": logits, "probs": torch.softmax(logits, 1)}


def exact(case, seed):
    op = case["op"]
    if op == "graph":
        got = _graph64(case, seed)
        return {k: v.cpu().numpy() for k, v in got.items()}
    t = _inputs(case, seed)
    d = [v.double() for v in t]
    if op == "binary":
        return [getattr(torch, case["fn"])(d[0], d[1])]
    if op == "qdq":
        if case["code"].startswith("float8"):
            return None                                 # the codes are not IEEE rounding of the quotient
        shape = [1, 1, 1]
        if case["axis"] >= 0:
            shape[case["axis"]] = -1
        s, z = d[1].reshape(shape), d[2].reshape(shape)
        lo, hi = (0, 255) if case["code"] == "uint8" else (-128, 127)
        code = torch.clamp(torch.round(d[0] / s) + z, lo, hi)
        return [code.to(TORCH_DTYPE[case["code"]]), (code - z) * s]
    if op == "softmax":
        return [torch.softmax(d[0], 1)]
    if op == "maxpool":
        return [torch.nn.functional.max_pool2d(d[0], case["k"], case["s"], case["p"])]
    if op == "gemm":
        return [d[0] @ (d[1].t().contiguous() if case["tb"] else d[1]) + d[2]]
    if op == "woq":
        return [d[0] @ (d[1] * d[2][:, None]).t().contiguous() + d[4]]
    return [_conv64(t[0], t[1], t[2], case["s"], case["k"] // 2, case["c"] if case["depthwise"] else 1)]
