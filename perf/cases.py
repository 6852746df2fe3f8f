"""What the framework is timed on: Float8 training steps and Float8 inference calls, each through the package's public
entry points (``convert_to_float8_training``, ``sync_float8_amax_and_scale_history``, ``quantize_to_float8``) as a
user's program makes them.

A training case is one step of ``linears`` layers k -> n that read the same m tokens (one projection, w1 / w3 of a
feed-forward block, q / k / v of an attention block): forward, backward with a given gradient, gradients set to None
before, as ``zero_grad()`` leaves them; with delayed scaling the bookkeeping of the step comes first.  An inference case
is one call of a quantised linear, or of the SiLU-gated feed-forward block of three of them, without gradients.
"""
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

import float8_experimental_amd as f8
from float8_experimental_amd.inference import ActivationCasting, QuantConfig, quantize_to_float8

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _train(name, m, k, n, linears=1, dtype="bf16", autocast=False, scaling="dynamic", bias=False):
    return {"name": name, "what": "train", "m": m, "k": k, "n": n, "linears": linears, "dtype": dtype, "autocast": autocast,
            "scaling": scaling, "bias": bias}


def _infer(name, m, k, n, block="linear", dtype="bf16", casting="dynamic", bias=False):
    return {"name": name, "what": "infer", "block": block, "m": m, "k": k, "n": n, "dtype": dtype, "casting": casting, "bias": bias}


def listed():
    return [
        # a small layer, the size of the unit tests and of a first experiment: latency and launches are all there is
        _train("train_small", 512, 1024, 1024),
        # one projection of a 4096-wide model at 2048 tokens: the first benchmark configuration
        _train("train_4096", 2048, 4096, 4096),
        # k and v projections of the 8B-shaped decoder at its 8192 tokens: grouped-query heads make them narrow
        _train("train_kv", 8192, 4096, 1024, linears=2),
        # w1 and w3 of the same decoder's feed-forward block: where such a model spends most of its step
        _train("train_ffn", 8192, 4096, 14336, linears=2),
        # the largest layer of the 70B shapes at 16384 tokens
        _train("train_70b_w13", 16384, 8192, 57344),
        # sizes that are multiples of nothing (the padding configuration)
        _train("train_ragged", 4099, 4097, 11007),
        # fp32 master weights and bias under bf16 autocast: a model that was never cast to bf16
        _train("train_autocast", 4096, 4096, 4096, dtype="fp32", autocast=True, bias=True),
        # delayed scaling of all three tensors, history 16, q / k / v shaped: sync, forward, backward
        _train("train_delayed", 2048, 4096, 4096, linears=3, scaling="delayed"),
        # decoding one token through one linear of a large model: the weight is read once, everything else is latency
        _infer("decode_linear", 1, 8192, 8192),
        # a decode batch through the feed-forward block of the inference tests (d = 4096, ffn = 14336)
        _infer("decode_ffn", 16, 4096, 14336, block="ffn"),
        # prefill of a prompt with calibrated (static) activation scale and a bias
        _infer("prefill_static", 2048, 4096, 14336, casting="static", bias=True),
        # weight-only quantisation, what it is bought for: few tokens and half the weight bytes
        _infer("decode_weight_only", 4, 4096, 14336, casting="weight_only"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size between lo and hi, spread over the logarithm; two of three are multiples of 128, as in most models."""
    v = _log_int(rng, lo, hi)
    return max(lo, v // 128 * 128) if rng.random() < 2 / 3 else v


def draw(rng):
    most = _flops(_train("", 16384, 8192, 57344))
    while True:
        if rng.random() < 0.6:
            dtype, autocast = rng.choice([("bf16", False)] * 5 + [("fp32", True)] * 2 + [("fp32", False), ("fp16", False)])
            case = _train("", _size(rng, 128, 16384), _size(rng, 512, 28672), _size(rng, 512, 28672), linears=rng.choice([1, 1, 2, 3]),
                          dtype=dtype, autocast=autocast, scaling=rng.choice(["dynamic", "dynamic", "delayed"]), bias=rng.random() < 0.25)
            if 3 * case["linears"] * case["n"] * max(case["m"], case["k"]) > 1.5e9:  # 2 GB a tensor, three sets of them
                continue
        else:
            m = _log_int(rng, 1, 64) if rng.random() < 0.6 else _size(rng, 128, 8192)
            case = _infer("", m, _size(rng, 1024, 16384), _size(rng, 1024, 16384), block=rng.choice(["linear", "linear", "ffn"]),
                          dtype=rng.choice(["bf16"] * 4 + ["fp16", "fp32"]), casting=rng.choice(["dynamic", "dynamic", "static", "weight_only"]),
                          bias=rng.random() < 0.25)
        if _flops(case) <= most:
            del case["name"]
            return case


class _Parallel(nn.Module):
    """Linear layers that read the same input."""

    def __init__(self, k, n, linears, bias, dtype):
        super().__init__()
        self.layers = nn.ModuleList(nn.Linear(k, n, bias=bias, device="cuda", dtype=dtype) for _ in range(linears))

    def forward(self, x):
        return [layer(x) for layer in self.layers]


class _FeedForward(nn.Module):
    def __init__(self, k, n, bias, dtype):
        super().__init__()
        self.w1 = nn.Linear(k, n, bias=bias, device="cuda", dtype=dtype)
        self.w3 = nn.Linear(k, n, bias=bias, device="cuda", dtype=dtype)
        self.w2 = nn.Linear(n, k, bias=bias, device="cuda", dtype=dtype)

    def forward(self, x):
        return self.w2(F.silu(self.w1(x)) * self.w3(x))


def _made(case, seed):
    """The model in high precision, its input and, to train, the gradients of its outputs."""
    torch.manual_seed(seed)
    m, k, n, dtype = case["m"], case["k"], case["n"], _DTYPES[case["dtype"]]
    normal = lambda *shape, dt=dtype, std=1.0: torch.empty(shape, device="cuda", dtype=dt).normal_(0.0, std)
    if case["what"] == "infer":
        model = _FeedForward(k, n, case["bias"], dtype) if case["block"] == "ffn" else nn.Linear(k, n, bias=case["bias"], device="cuda", dtype=dtype)
        return model, normal(m, k), None
    act = torch.bfloat16 if case["autocast"] else dtype  # what the layers before and after this one hand over
    model = _Parallel(k, n, case["linears"], case["bias"], dtype)
    return model, normal(m, k, dt=act), [normal(m, n, dt=act, std=1e-2) for _ in range(case["linears"])]


def prepare(case, seed):
    model, x, dys = _made(case, seed)
    if case["what"] == "infer":
        if case["casting"] == "static":  # as calibrated on activations that reach about 7
            quant = QuantConfig(ActivationCasting.STATIC, static_quantization_scale=torch.tensor([64.0], device="cuda"))
        else:
            quant = QuantConfig(ActivationCasting.DYNAMIC if case["casting"] == "dynamic" else ActivationCasting.WEIGHT_ONLY)
        return {"case": case, "model": quantize_to_float8(model, quant), "x": x}
    kind = f8.CastConfig(scaling_type=f8.ScalingType.DELAYED if case["scaling"] == "delayed" else f8.ScalingType.DYNAMIC)
    config = f8.Float8LinearConfig(cast_config_input=kind, cast_config_weight=kind, cast_config_grad_output=kind)
    model = f8.convert_to_float8_training(model, config=config)
    state = {"case": case, "model": model, "x": x.requires_grad_(), "dys": dys}
    if case["scaling"] == "delayed":
        _step(state)  # the first iteration, which initialises the amaxes, is behind a program that trains
    return state


def _step(state):
    case, model, x = state["case"], state["model"], state["x"]
    x.grad = None
    model.zero_grad()
    if case["scaling"] == "delayed" and model.layers[0].is_amax_initialized:
        f8.sync_float8_amax_and_scale_history(model)
    if case["autocast"]:
        with torch.autocast("cuda", dtype=torch.bfloat16):
            ys = model(x)
    else:
        ys = model(x)
    torch.autograd.backward(ys, state["dys"])
    out = {"y": ys, "dx": x.grad, "grads": [p.grad for p in model.parameters()]}
    if case["scaling"] == "delayed":
        out["buffers"] = list(model.buffers())
    return out


def run(state):
    if state["case"]["what"] == "train":
        return _step(state)
    with torch.no_grad():
        return state["model"](state["x"])


def _flops(case):
    if case["what"] == "train":
        return 6.0 * case["m"] * case["k"] * case["n"] * case["linears"]
    return 2.0 * case["m"] * case["k"] * case["n"] * (3 if case["block"] == "ffn" else 1)


def work(case):
    m, k, n = case["m"], case["k"], case["n"]
    size = 4 if case["dtype"] == "fp32" else 2
    if case["what"] == "infer":
        weights = n * k * (3 if case["block"] == "ffn" else 1)  # fp8: a byte each
        moved = weights + size * m * (2 * k if case["block"] == "ffn" else k + n)
    else:
        act = 2 if case["autocast"] else size
        # read: x, the weights, the gradients of the outputs; written: the outputs, the gradients of x and of the weights
        moved = act * 2 * m * k + case["linears"] * (act * 2 * m * n + size * 2 * n * k)
    return {"bytes": float(moved), "flops": _flops(case)}


def tolerance(case):
    # About four times what the path was measured to differ from the float64 products of the same fp8 operands, rounded
    # to the output's type (2-norm: bf16 2.0e-4, fp16 7e-5, fp32 1.2e-5 -- the matrix cores' alignment of products; one
    # ulp at most, two where a bias or another layer's gradient is added in that type).
    out = "bf16" if case["what"] == "train" and case["autocast"] else case["dtype"]
    rel, most = {"bf16": (8e-4, 0.03), "fp16": (3e-4, 4e-3), "fp32": (5e-5, 4e-4)}[out]
    if case["what"] == "infer" and case["casting"] == "weight_only" and out == "fp32":
        rel, most = 3e-6, 2e-5  # fp32 sums: 5.7e-7 and 2.8e-6
    if case["what"] == "infer" and case["block"] == "ffn":
        if case["casting"] == "weight_only":
            rel, most = 4 * rel, 2 * most  # three linears one behind the other: bf16 3.1e-4
        else:
            # the last bit of the hidden activations decides how some of them round to fp8 (bf16: 1.8e-3) and, with dynamic
            # scaling, may move their scale by one ulp, which rounds a tenth of them the other way (1.5e-2)
            rel, most = (0.02, 0.15) if case["casting"] == "dynamic" and out == "bf16" else (7e-3, 0.06)
    return {"rel": rel, "max": most}


def _dequantised(t, kind, scale=None, buffered=False):
    """t cast to fp8 as the path defines it, and back, in 64 bits: an operand of the exact products.  With the scale in a
    buffer (delayed, or given beforehand) its arithmetic and the product are in fp32, else in t's own type."""
    top = torch.finfo(kind).max
    buffered = buffered or scale is not None
    if scale is None:
        amax = t.abs().max()
        scale = (amax.float() if buffered else amax).clamp(min=1e-12).reciprocal() * top
        if t.dtype is torch.float16:
            scale = scale.clamp(max=65504.0)
        scale = scale.float()
    product = (t.float() if buffered else t) * scale
    return product.clamp(-top, top).to(kind).double() / scale.double()


def exact(case, seed):
    """The same outputs with every product of the fp8 operands in 64 bits; None for the buffers of delayed scaling."""
    model, x, dys = _made(case, seed)
    e4m3, e5m2 = torch.float8_e4m3fn, torch.float8_e5m2
    with torch.no_grad():
        if case["what"] == "infer":
            def linear(layer, x):
                if case["casting"] == "weight_only":  # the dequantised weight has the model's type, and no bias is added
                    return x.double() @ _dequantised(layer.weight, e4m3).to(x.dtype).double().t()
                static = torch.tensor([64.0], device="cuda") if case["casting"] == "static" else None
                y = _dequantised(x, e4m3, static) @ _dequantised(layer.weight, e4m3).t()
                return y if layer.bias is None else y + layer.bias.double()

            if case["block"] != "ffn":
                return linear(model, x)
            return linear(model.w2, F.silu(linear(model.w1, x).to(x.dtype)) * linear(model.w3, x).to(x.dtype))
        delayed = case["scaling"] == "delayed"
        x8 = _dequantised(x, e4m3, buffered=delayed)
        ys, dx, grads = [], 0.0, []
        for layer, dy in zip(model.layers, dys):
            w8, dy8 = _dequantised(layer.weight, e4m3, buffered=delayed), _dequantised(dy, e5m2, buffered=delayed)
            y = x8 @ w8.t()
            ys.append(y if layer.bias is None else y + layer.bias.to(x.dtype).double())
            dx = dx + dy8 @ w8
            grads.append(dy8.t() @ x8)
            if layer.bias is not None:
                grads.append(dy.double().sum(0))
        out = {"y": ys, "dx": dx, "grads": grads}
        if delayed:
            out["buffers"] = [None] * (9 * case["linears"])
        return out
