"""The calls whose speed counts: quantised and fp16 linears through the package's public entry points.

A case is one of four kinds:

  linear   one eager call of a linear on activations and weights in hand (`op` names the
           entry point): image and text tokens of a diffusion transformer, prompt prefill,
           a batch of decode rows;
  step     the linears of `layers` decoder layers for a few rows, captured once in a HIP
           graph and replayed, as a serving loop runs a decode step;
  convrot  one ConvRot layer object of a diffusion transformer;
  fp16     the two fp16 linears, a depth decoder's GEMV and a diffusion transformer's GEMM.

Activations are N(0, 1) in the model's type. Weight codes are those of Gaussian weights
quantised per output row by their largest magnitude, scales lie in 0.002 .. 0.02.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "omni-rs_amd"))
import omni_int8  # noqa: E402
from omni_int8 import convrot, f16  # noqa: E402

DEVICE = "cuda"
GROUP = 128  # int4 values per scale
F16 = {"f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # One token of a TTS depth decoder: the smallest call, where latency counts.
        {"name": "f16_depth_gemv", "kind": "fp16", "op": "gemv", "rows": 1, "width": 8192, "columns": 1024},
        # A decode step of eight sequences through one W8A8 layer of a 7B decoder.
        {"name": "int8_step_8", "kind": "step", "op": "int8", "rows": 8, "hidden": 4096, "ffn": 14336, "kv": 1024,
         "layers": 1},
        # The text tokens of a diffusion transformer's QKV projection, with its bias, in the model's type.
        {"name": "int8_text_77", "kind": "linear", "op": "int8_bias", "rows": 77, "width": 3072, "columns": 9216,
         "x": "f16"},
        # The operator at the reference's benchmark shape: 256 rows, long K.
        {"name": "int8_256", "kind": "linear", "op": "int8", "rows": 256, "width": 12288, "columns": 4096, "x": "f16"},
        # The image tokens of a 1024 x 1024 picture, MLP up.
        {"name": "int8_image", "kind": "linear", "op": "int8", "rows": 4096, "width": 3072, "columns": 12288,
         "x": "f16"},
        # Image and text tokens through a ConvRot MLP down projection.
        {"name": "convrot_down", "kind": "convrot", "rows": 4352, "width": 12288, "columns": 3072, "x": "f16"},
        # One sequence's decode step through four layers of a small vision-language model, weight-only int8.
        {"name": "w8a16_step_1", "kind": "step", "op": "w8a16", "rows": 1, "hidden": 1536, "ffn": 8960, "kv": 256,
         "layers": 4},
        # A batch of 24 decode rows through a 7B MLP up projection.
        {"name": "w8a16_batch_24", "kind": "linear", "op": "w8a16", "rows": 24, "width": 4096, "columns": 14336},
        # A prompt of 1000 tokens through a small model's MLP up projection.
        {"name": "w8a16_prompt_1000", "kind": "linear", "op": "w8a16", "rows": 1000, "width": 1536, "columns": 8960},
        # One sequence's decode step through a packed-int4 layer.
        {"name": "w4a16_step_1", "kind": "step", "op": "w4a16", "rows": 1, "hidden": 3584, "ffn": 18944, "kv": 512,
         "layers": 1},
        # A prompt of 500 tokens through the same model's MLP up projection.
        {"name": "w4a16_prompt_500", "kind": "linear", "op": "w4a16", "rows": 500, "width": 3584, "columns": 18944},
        # The image tokens through an fp16 projection of a diffusion transformer.
        {"name": "f16_dit_gemm", "kind": "fp16", "op": "gemm", "rows": 4096, "width": 4096, "columns": 12288},
    ]


LARGEST = 2.0 * 4096 * 4096 * 12288  # the largest listed case's operations


def _spread(rng, low, high, step=1):
    """A multiple of `step` from low to high, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(v / step)) * step))


def _draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "step", "step", "step", "convrot", "fp16"])
    # Most widths are multiples of 64; vision towers have ragged ones (4304, 1152 + 16 ...).
    step = rng.choice([64, 64, 64, 16])
    if kind == "linear":
        op = rng.choice(["int8", "int8_bias", "w8a16", "w4a16"])
        if op == "w4a16":
            step = GROUP
        return {"kind": kind, "op": op, "rows": _spread(rng, 5, 4352), "width": _spread(rng, 1024, 14336, step),
                "columns": _spread(rng, 1024, 18944, rng.choice([64, 64, 4, 1])),
                **({"x": rng.choice(["f16", "f32"])} if op.startswith("int8") else {})}
    if kind == "step":
        op = rng.choice(["int8", "w8a16", "w4a16"])
        hidden = _spread(rng, 1536, 4096, GROUP if op == "w4a16" else step)
        ffn = int(hidden * rng.uniform(2.5, 5.8)) // 128 * 128
        return {"kind": kind, "op": op, "rows": _spread(rng, 1, 48 if op == "int8" else 16), "hidden": hidden,
                "ffn": ffn, "kv": rng.choice([256, 512, 1024]), "layers": 1 if hidden > 2560 else rng.choice([1, 2, 4])}
    if kind == "convrot":
        return {"kind": kind, "rows": _spread(rng, 16, 4352), "width": _spread(rng, 1536, 12288, 256),
                "columns": _spread(rng, 1536, 12288, 16), "x": rng.choice(["f16", "f16", "f32"])}
    if rng.random() < 0.5:
        return {"kind": kind, "op": "gemv", "rows": _spread(rng, 1, 64), "width": _spread(rng, 1024, 8192, 32),
                "columns": _spread(rng, 512, 4096, 8)}
    return {"kind": kind, "op": "gemm", "rows": _spread(rng, 256, 4352), "width": _spread(rng, 4096, 12288, 64),
            "columns": _spread(rng, 4096, 12288, 64)}


def draw(rng):
    while True:
        case = _draw(rng)
        if work(case)["flops"] <= LARGEST:
            return case


def _linears(case):
    """(width, columns) of each linear of a pass."""
    if case["kind"] != "step":
        return [(case["width"], case["columns"])]
    h, f, kv = case["hidden"], case["ffn"], case["kv"]
    return [(h, h + 2 * kv), (h, h), (h, 2 * f), (f, h)] * case["layers"]


def _op(case):
    return {"convrot": "convrot", "fp16": "fp16"}.get(case["kind"]) or case["op"]


def work(case):
    op, rows = _op(case), case["rows"]
    x = 4 if case.get("x") == "f32" else 2
    y = 4 if op == "int8" else 2
    total = {"bytes": 0.0, "flops": 0.0}
    for k, n in _linears(case):
        weights = {"fp16": 2.0 * k, "w4a16": 0.5 * k + 2.0 * (k // GROUP)}.get(op, 1.0 * k) * n
        vectors = {"int8": 8, "convrot": 8, "int8_bias": 12, "w8a16": 2}.get(op, 0) * n
        total["bytes"] += x * rows * k + weights + vectors + y * rows * n
        total["flops"] += 2.0 * rows * k * n
    return total


def tolerance(case):
    op = _op(case)
    if op in ("int8", "int8_bias"):
        return "exact"  # codes and sums are integers, the epilogue is three f32 operations in a given order
    # f32 sums rounded once to f16 (ConvRot: the rotation's sums in another order also move a
    # code in some ten thousand to its neighbour): 2.1e-4 off the 64-bit result.
    return {"rel": 1e-3}


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _codes(g, n, k, top):
    w = torch.empty((n, k), dtype=torch.int8, device=DEVICE)
    part = max(1, (1 << 25) // k)
    for i in range(0, n, part):
        v = torch.randn((min(part, n - i), k), generator=g, device=DEVICE)
        w[i:i + part] = (v * (top / v.abs().amax(1, keepdim=True))).round_().to(torch.int8)
    return w


def _uniform(g, n, dtype):
    return (torch.rand(n, generator=g, device=DEVICE) * 0.018 + 0.002).to(dtype)


def _inputs(g, case, k, n):
    """Activations and weights of one linear, and the weight's codes for exact()."""
    op, rows = _op(case), case["rows"]
    x = torch.randn((rows, k), generator=g, device=DEVICE)
    if op == "convrot":  # a hundredth of the channels are outliers
        x = torch.where(torch.rand(k, generator=g, device=DEVICE) < 0.01, x * 20, x)
    x = x.to(F16[case.get("x", "f16")])
    if op == "fp16":
        return {"x": x, "w": (torch.randn((n, k), generator=g, device=DEVICE) * 0.02).half().t()}
    if op == "w4a16":
        q = _codes(g, n, k, 7) + 8
        packed = (q[:, 0::2] | (q[:, 1::2] << 4)).to(torch.uint8)
        scale = _uniform(g, n * (k // GROUP), torch.bfloat16).reshape(n, k // GROUP)
        return {"x": x, "w": packed, "scale": scale}
    w = _codes(g, n, k, 127)
    if op == "w8a16":
        return {"x": x, "w": w, "scale": _uniform(g, n, torch.float16)}
    zero = torch.randint(-3, 4, (n,), generator=g, device=DEVICE, dtype=torch.int32)
    v = {"x": x, "w": w, "scale": _uniform(g, n, torch.float32), "zero": zero}
    if op == "int8_bias":
        v["bias"] = torch.randn(n, generator=g, device=DEVICE)
    return v


def _call(op, v):
    if op == "int8":
        return omni_int8.try_int8_gemm(v["x"], v["packed"], v["scale"], v["zero"])
    if op == "int8_bias":
        codes, row_scale, row_sum = omni_int8.quantize_rows(v["x"])
        return omni_int8.w8a8_gemm(codes, row_scale, row_sum, v["w"], v["scale"], v["zero"], v["bias"], torch.float16)
    if op == "w8a16":
        return omni_int8.w8a16_linear(v["x"], v["w"], v["scale"])
    return omni_int8.w4a16_linear(v["x"], v["w"], v["scale"], None, GROUP)


def prepare(case, seed):
    g, op = _generator(seed), _op(case)
    every = [_inputs(g, case, k, n) for k, n in _linears(case)]
    for v in every:
        if op == "int8":
            v["packed"] = omni_int8.pack_i8(v["w"])
    state = {"kind": case["kind"], "op": op, "every": every}
    if case["kind"] == "convrot":
        v = every[0]
        state["layer"] = convrot.Int8Linear(case["width"], case["columns"], omni_int8.pack_i8(v["w"]), v["scale"],
                                            v["zero"])
    if case["kind"] == "fp16":
        state["linear"] = f16.depth_try_linear if case["op"] == "gemv" else f16.tensorops_try_linear
    if case["kind"] == "step":
        torch.cuda.synchronize()
        for v in every:  # kernels are loaded outside the capture
            _call(op, v)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["outputs"] = [_call(op, v) for v in every]
    return state


def run(state):
    if state["kind"] == "step":
        state["graph"].replay()
        return state["outputs"]
    v = state["every"][0]
    if state["kind"] == "convrot":
        return state["layer"](v["x"])
    if state["kind"] == "fp16":
        return state["linear"](v["x"], v["w"])
    return _call(state["op"], v)


def _exact(op, v):
    x = v["x"]
    if op == "fp16":
        return x.double() @ v["w"].double()
    if op == "w8a16":
        return (x.double() @ v["w"].double().t()) * v["scale"].double()
    if op == "w4a16":
        q = torch.stack((v["w"] & 15, v["w"] >> 4), dim=-1).reshape(v["w"].shape[0], -1).double() - 8.0
        return x.double() @ (q * v["scale"].double().repeat_interleave(GROUP, dim=1)).t()
    x = x.float()
    if op == "convrot":
        h4 = torch.ones((4, 4), dtype=torch.float64, device=DEVICE)
        for i in range(4):
            h4[i, 3 - i] = -1.0
        h = torch.kron(torch.kron(h4, h4), torch.kron(h4, h4)) / 16.0
        x = (x.double().reshape(-1, 256) @ h).reshape(x.shape)
    # Codes are whole numbers by contract: the peak over 127, then round half away from zero.
    # The scale and the quotients are f32 values, correctly rounded (here by way of f64).
    row_scale = (x.abs().amax(1, keepdim=True).double() / 127.0).float()
    q = x.double() / row_scale.double()
    q = q if op == "convrot" else q.float()
    codes = ((q.abs() + 0.5).floor() * q.sign()).clamp(-128, 127).double()
    acc = codes @ v["w"].double().t() - codes.sum(1, keepdim=True) * v["zero"].double()
    out = acc * row_scale.double() * v["scale"].double()
    return out + v["bias"].double() if "bias" in v else out


def exact(case, seed):
    g, op = _generator(seed), _op(case)
    outs = [_exact(op, _inputs(g, case, k, n)) for k, n in _linears(case)]
    return outs if case["kind"] == "step" else outs[0]
