"""The work that programs built on rotalabs_accel have it do, as cases to time.

A case is a dict of plain values; ``op`` names the entry point it goes
through:

* ``gemm``      ``int8_gemm``: one projection of a served model.
* ``linear``    ``Int8Linear`` with a bias, at sizes that are no multiples of anything.
* ``linear32``  ``QuantizedLinear`` with its fp32 bias, hence fp32 activations:
                what ``quantize_model`` makes of an fp32 model.
* ``mlp``       ``Int8SwiGLUMLP`` (the decoder MLP with its RMSNorm), or with a
                bias ``Int8SwiGLU``.
* ``w8a8``      ``quantized_matmul.int8_gemm(use_cublas=True)``.
* ``kv``        ``QuantizedTensor`` and its ``dequantize``: a KV block put away and read back.
* ``rowops``    the unfused ops of a decoder layer whose projections are not int8:
                ``rmsnorm_residual_fused`` and ``swiglu_fused`` (``swiglu_with_bias``
                where the projections leave the bias to it).
* ``quantize``  ``quantize_weight_per_channel``: a checkpoint's weight on load.

Weights are int8 values of a normal distribution whose row maximum is 127,
with scales of 11 significant bits, so that quantising ``q * s`` gives back
``q`` and ``s`` exactly.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "rotalabs-accel_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

DEVICE = "cuda"
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}
EPS = 1e-6


def listed():
    return [
        # One token's projection, hidden to hidden: the shortest call a decode step makes.
        {"name": "gemm_decode", "op": "gemm", "M": 1, "K": 4096, "N": 4096, "dtype": "float16", "bias": False},
        # A decode step of 64 sequences through an FFN projection.
        {"name": "gemm_batch", "op": "gemm", "M": 64, "K": 4096, "N": 11008, "dtype": "bfloat16", "bias": False},
        # A prompt of 2048 tokens through the same projection.
        {"name": "gemm_prefill", "op": "gemm", "M": 2048, "K": 4096, "N": 11008, "dtype": "float16", "bias": False},
        # A head or adapter whose sizes nobody rounded up, over a short prompt.
        {"name": "linear_ragged", "op": "linear", "M": 77, "K": 1000, "N": 4101, "dtype": "float16"},
        # A layer of an fp32 model converted by quantize_model, over a few short texts.
        {"name": "linear_fp32", "op": "linear32", "M": 512, "K": 4096, "N": 4096},
        # The decoder MLP of a large model in a decode step of 17 sequences, residual stream given.
        {"name": "mlp_decode", "op": "mlp", "M": 17, "H": 8192, "I": 28672, "dtype": "bfloat16", "residual": True,
         "bias": False},
        # The MLP of a smaller one over a mixed batch: some decoding sequences and a piece of a prompt.
        {"name": "mlp_mixed", "op": "mlp", "M": 200, "H": 4096, "I": 11008, "dtype": "bfloat16", "residual": True,
         "bias": False},
        # The large model's MLP over a long prompt.
        {"name": "mlp_prefill", "op": "mlp", "M": 4096, "H": 8192, "I": 28672, "dtype": "bfloat16",
         "residual": False, "bias": False},
        # A piece of a prompt with int8 activations too.
        {"name": "w8a8_chunk", "op": "w8a8", "M": 512, "K": 4096, "N": 11008, "dtype": "float16", "bias": False},
        # One layer's keys of 8 sequences, 32 heads, 4096 tokens: put away and read back.
        {"name": "kv_block", "op": "kv", "B": 8, "heads": 32, "tokens": 4096, "dim": 128, "bits": 8,
         "dtype": "bfloat16"},
        # The elementwise ops of a decoder layer over a prompt of 4096 tokens.
        {"name": "layer_rowops", "op": "rowops", "M": 4096, "H": 4096, "I": 11008, "dtype": "bfloat16",
         "weight": "bfloat16", "bias": False},
        # One projection of an fp16 checkpoint quantised on load.
        {"name": "quantize_load", "op": "quantize", "N": 11008, "K": 4096, "dtype": "float16"},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of ``step`` in [lo, hi], spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi // step * step, max(-(-lo // step) * step, int(round(v / step)) * step))


def draw(rng):
    op = rng.choice(("gemm", "gemm", "gemm", "linear", "linear32", "mlp", "mlp", "w8a8", "kv", "rowops", "quantize"))
    half = rng.choice(("float16", "bfloat16"))
    if op == "gemm":
        return {"op": op, "M": _log(rng, 1, 4096), "K": _log(rng, 1024, 16384, 64), "N": _log(rng, 1000, 16384),
                "dtype": half, "bias": rng.random() < 0.3}
    if op == "linear":
        return {"op": op, "M": _log(rng, 1, 512), "K": _log(rng, 300, 4100), "N": _log(rng, 300, 8200), "dtype": half}
    if op == "linear32":
        return {"op": op, "M": _log(rng, 1, 512), "K": _log(rng, 300, 4096, rng.choice((1, 64))),
                "N": _log(rng, 300, 4096)}
    if op == "mlp":
        return {"op": op, "M": _log(rng, 1, 2048), "H": _log(rng, 1024, 8192, 128), "I": _log(rng, 2048, 28672, 32),
                "dtype": half, "residual": rng.random() < 0.5, "bias": rng.random() < 0.25}
    if op == "w8a8":
        return {"op": op, "M": _log(rng, 17, 4096), "K": _log(rng, 1024, 11008, 64), "N": _log(rng, 1000, 16384),
                "dtype": half, "bias": rng.random() < 0.3}
    if op == "kv":
        return {"op": op, "B": _log(rng, 1, 8), "heads": rng.choice((8, 16, 32)), "tokens": _log(rng, 1, 4096),
                "dim": rng.choice((64, 80, 96, 128)), "bits": rng.choice((8, 8, 4)), "dtype": half}
    if op == "rowops":
        step = rng.choice((1, 8, 64))
        return {"op": op, "M": _log(rng, 1, 4096), "H": _log(rng, 1000, 8192, step), "I": _log(rng, 2048, 16384, step),
                "dtype": half, "weight": rng.choice((half, "float32")), "bias": rng.random() < 0.3}
    return {"op": op, "N": _log(rng, 1000, 11008), "K": _log(rng, 300, 8192, rng.choice((1, 8, 64))),
            "dtype": rng.choice(("float16", "bfloat16", "float32"))}


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _normal(g, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEVICE, dtype=torch.float32) * std).to(dtype)


def _weight(g, n, k):
    """(q, s): int8 [n, k] with a 127 in each row, fp32 [n] near 0.02 / 32."""
    q = torch.randn(n, k, generator=g, device=DEVICE).mul_(32.0).round_().clamp_(-127, 127).to(torch.int8)
    at = torch.randint(0, k, (n, 1), generator=g, device=DEVICE)
    q.scatter_(1, at, torch.full((n, 1), 127, dtype=torch.int8, device=DEVICE))
    s = torch.randint(1024, 2048, (n,), generator=g, device=DEVICE).float() * 2.0 ** -21
    return q, s


def _linear_of(cls, q, s, bias):
    lin = torch.nn.Linear(q.shape[1], q.shape[0], bias=True, device=DEVICE, dtype=torch.float32)
    lin.weight.data.copy_(q.float() * s[:, None])
    lin.bias.data.copy_(bias)
    return cls.from_linear(lin)


def _inputs(case, seed):
    """What a case is made from, as plain tensors: the same for prepare() and exact()."""
    g, op = _gen(seed), case["op"]
    dt = DTYPES[case.get("dtype", "float32")]
    if op in ("gemm", "linear", "linear32", "w8a8"):
        d = {"x": _normal(g, case["M"], case["K"], dtype=dt)}
        d["q"], d["s"] = _weight(g, case["N"], case["K"])
        if case.get("bias", True):
            # (an Int8Linear's bias is fp16, whatever the activations are)
            bdt = torch.float16 if op == "linear" else dt
            d["b"] = _normal(g, case["N"], dtype=bdt, std=0.1)
        return d
    if op == "mlp":
        H, inter = case["H"], case["I"]
        d = {"x": _normal(g, case["M"], H, dtype=dt)}
        d["norm"] = (1.0 + 0.01 * _normal(g, H)).to(dt)
        if case["residual"]:
            d["r"] = _normal(g, case["M"], H, dtype=dt)
        d["q_gu"], d["s_gu"] = _weight(g, 2 * inter, H)
        d["q_d"], d["s_d"] = _weight(g, H, inter)
        if case["bias"]:
            d["b_gu"] = _normal(g, 2 * inter, dtype=torch.float16, std=0.1)
            d["b_d"] = _normal(g, H, dtype=torch.float16, std=0.1)
        return d
    if op == "kv":
        t = _normal(g, case["B"], case["heads"], case["tokens"], case["dim"])
        # keys have a few channels that are larger than the others
        t *= 1.0 + 4.0 * (torch.rand(case["heads"], 1, case["dim"], generator=g, device=DEVICE) < 0.03)
        return {"t": t.to(dt)}
    if op == "rowops":
        wdt = DTYPES[case["weight"]]
        d = {"x": _normal(g, case["M"], case["H"], dtype=dt), "r": _normal(g, case["M"], case["H"], dtype=dt),
             "w": (1.0 + 0.01 * _normal(g, case["H"])).to(wdt),
             "gate": _normal(g, case["M"], case["I"], dtype=dt), "up": _normal(g, case["M"], case["I"], dtype=dt)}
        if case["bias"]:
            d["bg"] = _normal(g, case["I"], dtype=dt, std=0.1)
            d["bu"] = _normal(g, case["I"], dtype=dt, std=0.1)
        return d
    return {"w": _normal(g, case["N"], case["K"], dtype=dt, std=0.02)}


def _mlp_module(case, d):
    import rotalabs_accel as ra
    inter = case["I"]
    with torch.device(DEVICE):
        if case["bias"]:
            m = ra.Int8SwiGLU(case["H"], inter, bias=True)
            m.bias_gate_up.data, m.bias_down.data = d["b_gu"], d["b_d"]
        else:
            m = ra.Int8SwiGLUMLP(case["H"], inter, eps=EPS, norm_dtype=DTYPES[case["dtype"]])
            m.norm_weight.data = d["norm"]
    # the int8 buffers as a saved model holds them
    m.weight_gate_up, m.scale_gate_up = d["q_gu"], d["s_gu"]
    m.weight_down, m.scale_down = d["q_d"], d["s_d"]
    m._quantized = True
    return m.requires_grad_(False)


def prepare(case, seed):
    import rotalabs_accel as ra
    d = _inputs(case, seed)
    state = {"case": case, "in": d}
    if case["op"] == "linear":
        state["module"] = _linear_of(ra.Int8Linear, d["q"], d["s"], d["b"].float()).requires_grad_(False)
    elif case["op"] == "linear32":
        state["module"] = _linear_of(ra.QuantizedLinear, d["q"], d["s"], d["b"]).to(DEVICE).requires_grad_(False)
    elif case["op"] == "mlp":
        state["module"] = _mlp_module(case, d)
    if "module" in state:
        for k in ("q", "s", "b"):
            d.pop(k, None)
    return state


def run(state):
    import rotalabs_accel as ra
    case, d = state["case"], state["in"]
    op = case["op"]
    if op == "gemm":
        return ra.int8_gemm(d["x"], d["q"], d["s"], d.get("b"))
    if op in ("linear", "linear32"):
        return state["module"](d["x"])
    if op == "mlp":
        if case["bias"]:
            return state["module"](d["x"])
        return state["module"](d["x"], d.get("r"))
    if op == "w8a8":
        from rotalabs_accel.kernels import quantized_matmul
        return quantized_matmul.int8_gemm(d["x"], d["q"], d["s"], d.get("b"), use_cublas=True)
    if op == "kv":
        from rotalabs_accel.speculative.kv_compression import QuantizedTensor
        t = QuantizedTensor(d["t"], bits=case["bits"], per_channel=True)
        return {"data": t.data, "scale": t.scale, "values": t.dequantize()}
    if op == "rowops":
        h = ra.rmsnorm_residual_fused(d["x"], d["r"], d["w"], EPS)
        if case["bias"]:
            from rotalabs_accel.kernels.swiglu import swiglu_with_bias
            return {"norm": h, "act": swiglu_with_bias(d["gate"], d["up"], d["bg"], d["bu"])}
        return {"norm": h, "act": ra.swiglu_fused(d["gate"], d["up"])}
    q, s = ra.quantize_weight_per_channel(d["w"])
    return {"q": q, "s": s}


def _size(dtype):
    return DTYPES[dtype].itemsize


def work(case):
    op = case["op"]
    e = _size(case.get("dtype", "float32"))
    if op in ("gemm", "linear", "linear32", "w8a8"):
        M, K, N = case["M"], case["K"], case["N"]
        b = (2 if op == "linear" else e) * N if case.get("bias", True) else 0
        return {"bytes": N * K + 4 * N + e * M * K + e * M * N + b, "flops": 2 * M * N * K}
    if op == "mlp":
        M, H, inter = case["M"], case["H"], case["I"]
        b = 2 * (2 * inter + H) if case["bias"] else e * H
        return {"bytes": 3 * H * inter + 8 * inter + 4 * H + b + e * M * H * (3 if case["residual"] and not case["bias"] else 2),
                "flops": 6 * M * H * inter}
    if op == "kv":
        n = case["B"] * case["heads"] * case["tokens"] * case["dim"]
        rows = n // case["dim"]
        # encode: values in, codes and scales out; decode: the other way round
        return {"bytes": 2 * (e * n + n + e * rows), "flops": 0}
    if op == "rowops":
        M, H, inter = case["M"], case["H"], case["I"]
        wide = 4 if case["weight"] == "float32" else e
        return {"bytes": 2 * e * M * H + wide * (H + M * H) + 3 * e * M * inter + (2 * e * inter if case["bias"] else 0),
                "flops": 0}
    N, K = case["N"], case["K"]
    return {"bytes": e * N * K + N * K + 4 * N, "flops": 0}


def tolerance(case):
    """About four times what the path differs by from the same in 64 bits."""
    op = case["op"]
    if op in ("kv", "quantize"):
        return "exact"  # codes, scales and values are specified bit for bit
    if op == "linear32":
        return {"rel": 1e-6}
    # One rounding to 16 bits is 2e-4 (fp16) or 1.7e-3 (bf16) of the norm; the
    # RMSNorm of a sum has three on its way (2.9e-3 in bf16) and an MLP block
    # more (5.7e-3).
    if op == "mlp":
        return {"rel": 3e-3 if case["dtype"] == "float16" else 2.2e-2}
    if op == "rowops":
        return {"rel": 1.5e-3 if case["dtype"] == "float16" else 1.2e-2}
    return {"rel": 9e-4 if case["dtype"] == "float16" else 7e-3}


def _matmul64(x, q, s, b=None):
    """x @ (q * s).T + b in 64 bits, some rows of q at a time."""
    out = torch.empty(x.shape[0], q.shape[0], dtype=torch.float64, device=x.device)
    x = x.double()
    for i in range(0, q.shape[0], 8192):
        out[:, i:i + 8192] = (x @ q[i:i + 8192].double().t()) * s[i:i + 8192].double()
    return out if b is None else out + b.double()


def _rmsnorm64(v, w):
    return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS) * w.double()


def _silu64(v):
    return v / (1.0 + torch.exp(-v))


def exact(case, seed):
    d, op = _inputs(case, seed), case["op"]
    if op in ("gemm", "linear", "linear32"):
        return _matmul64(d["x"], d["q"], d["s"], d.get("b"))
    if op == "mlp":
        inter = case["I"]
        if case["bias"]:
            v = d["x"].double()
        else:
            v = _rmsnorm64(d["x"].double() + (d["r"].double() if "r" in d else 0.0), d["norm"])
        gu = _matmul64(v, d["q_gu"], d["s_gu"], d.get("b_gu"))
        return _matmul64(_silu64(gu[:, :inter]) * gu[:, inter:], d["q_d"], d["s_d"], d.get("b_d"))
    if op == "w8a8":
        # the activations' codes as the route defines them, each step rounded to their type
        dt = d["x"].dtype

        def rnd(v):
            return v.to(dt).double()

        top = d["x"].abs().amax(1, keepdim=True).double().clamp(min=1e-5)
        codes = rnd(d["x"].double() * rnd(rnd(1.0 / top) * 127.0)).round().clamp(-128, 127)
        if case["M"] < 17:
            return _matmul64(d["x"], d["q"], d["s"], d.get("b"))
        y = (codes @ d["q"].double().t()) * rnd(top / 127.0) * d["s"].double()
        return y + d["b"].double() if "b" in d else y
    if op == "kv":
        t, top = d["t"].double(), 2 ** (case["bits"] - 1) - 1
        s = (t.abs().amax(-1, keepdim=True) / top).clamp(min=1e-8)
        # codes are whole values; the values read back follow the stored scale's own rounding
        return {"data": None, "scale": s, "values": None}
    if op == "rowops":
        gate, up = d["gate"].double(), d["up"].double()
        if case["bias"]:
            gate, up = gate + d["bg"].double(), up + d["bu"].double()
        return {"norm": _rmsnorm64(d["x"].double() + d["r"].double(), d["w"]), "act": _silu64(gate) * up}
    s = d["w"].double().abs().amax(1) / 127.0
    return {"q": None, "s": s}
