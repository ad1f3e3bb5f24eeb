"""The native host path (csrc/host/ra_host.cpp): it declines what it does not
take, and what it takes gives the Python path's bits."""
import importlib

import pytest
import torch

import rotalabs_accel as ra
from rotalabs_accel import _backend
from rotalabs_accel.kernels import quantized_matmul as qm
from rotalabs_accel.kernels.swiglu import swiglu_with_bias
from rotalabs_accel.speculative import QuantizedTensor

MODULES = ["rotalabs_accel.kernels." + m for m in ("gemm", "mlp", "normalization", "activations", "swiglu",
                                                   "quantized_matmul")] + \
          ["rotalabs_accel.quantization.symmetric", "rotalabs_accel.speculative.kv_compression"]


def test_built_and_declines_cpu_tensors():
    _backend.load()
    assert _backend.host is not None, "the host extension is built with the library"
    x, q, s = torch.randn(2, 32), torch.zeros(8, 32, dtype=torch.int8), torch.ones(8)
    assert _backend.host.gemm(x, q, s, None) is None
    assert _backend.host.gemm(x, q, s) is None            # argument count
    assert _backend.host.swiglu(x, None) is None and _backend.host.quantize("x") is None
    assert _backend.host.rmsnorm(x, None, s, 1) is None   # eps no float


def _pairs(fn, monkeypatch):
    """fn() through the native path and through the Python path."""
    a = fn()
    with monkeypatch.context() as m:
        for name in MODULES:
            m.setattr(importlib.import_module(name), "_host", None)
        b = fn()
    return a, b


def _case(M, K, N, dt, gpu):
    g = torch.Generator().manual_seed(M + K + N)
    return (torch.randn(M, K, generator=g).to(dt).to(gpu),
            torch.randint(-127, 128, (N, K), generator=g).to(torch.int8).to(gpu),
            (torch.rand(N, generator=g) * 1e-2).to(gpu))


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
def test_same_bits_as_the_python_path(gpu, monkeypatch, dt):
    print(f"  host path {dt}", flush=True)
    for M, K, N in [(1, 64, 48), (5, 8192, 512), (70, 333, 77), (40, 2048, 8192), (3, 100, 20)]:
        x, q, s = _case(M, K, N, dt, gpu)
        b = torch.randn(N, device=gpu)
        forms = {
            "plain": lambda: ra.int8_gemm(x, q, s),
            "3-D": lambda: ra.int8_gemm(x.view(1, M, K), q, s, b.to(dt)),
            "strided x": lambda: ra.int8_gemm(torch.cat([x, x], 1)[:, :K], q, s, b),
            "transposed weight": lambda: ra.int8_gemm(x, q.t().contiguous().t(), s),
            "fp64 scale": lambda: ra.int8_gemm(x, q, s.double(), b.half()),
            "bias [1, N]": lambda: ra.int8_gemm(x, q, s, b[None]),
            "bias [1]": lambda: ra.int8_gemm(x, q, s, b[:1]),
            "no rows": lambda: ra.int8_gemm(x[:0], q, s),
            "gate/up": lambda: ra.int8_gateup_swiglu(x, q[:N // 2 * 2], s[:N // 2 * 2]),
            "odd address": lambda: ra.int8_gemm(torch.cat([x[0, :1], x.flatten()])[1:].view(M, K), q, s),
        }
        for name, fn in forms.items():
            a, p = _pairs(fn, monkeypatch)
            assert a.shape == p.shape and a.dtype == p.dtype and torch.equal(a, p), (name, M, K, N)
        w = torch.randn(K, device=gpu)
        for wt in (w.to(dt), w, w.half()):
            for fn in (lambda: ra.rmsnorm(x, wt), lambda: ra.rmsnorm_residual_fused(x, x.float(), wt, 1e-5),
                       lambda: ra.rmsnorm(x.t().contiguous().t(), wt, 1)):
                a, p = _pairs(fn, monkeypatch)
                assert a.dtype == p.dtype and torch.equal(a, p)
        for fn in (lambda: ra.swiglu_fused(x, x), lambda: ra.swiglu_fused(x.t(), x.t()),
                   lambda: swiglu_with_bias(x, x, w, w.half()), lambda: swiglu_with_bias(x, x, w, w),
                   lambda: ra.quantize_weight_per_channel(x)[0], lambda: ra.quantize_weight_per_channel(x.t())[1],
                   lambda: QuantizedTensor(x, 4).scale, lambda: QuantizedTensor(x[None]).dequantize(),
                   lambda: QuantizedTensor(x, 8, per_channel=False).dequantize()):
            a, p = _pairs(fn, monkeypatch)
            assert a.shape == p.shape and a.dtype == p.dtype and torch.equal(a, p)
        if dt != torch.float32 and M >= 17:
            a, p = _pairs(lambda: qm.int8_gemm(x, q, s, b, use_cublas=True), monkeypatch)
            assert torch.equal(a, p)


@pytest.mark.gpu
def test_refusals_stay(gpu):
    x, q, s = _case(4, 64, 32, torch.float16, gpu)
    print("  host path refusals", flush=True)
    for bad in (lambda: ra.int8_gemm(x, q.float(), s), lambda: ra.int8_gemm(x[:, :32], q, s),
                lambda: ra.int8_gemm(x, q, s[:3]), lambda: ra.rmsnorm(x, s), lambda: ra.swiglu_fused(x, x[:2])):
        with pytest.raises(AssertionError):
            bad()
    for bad in (lambda: ra.int8_gemm(x, q, s, torch.zeros(7, device=gpu)), lambda: ra.swiglu_fused(x, x.float()),
                lambda: ra.int8_gemm(x, q, s, torch.zeros(32))):
        with pytest.raises(RuntimeError):
            bad()
    with pytest.raises(TypeError):
        ra.int8_gemm(x.double(), q, s)


@pytest.mark.gpu
@pytest.mark.parametrize("residual", [False, True])
def test_mlp_same_bits_and_on_its_stream(gpu, monkeypatch, residual):
    """The whole block in one native call, also on another stream (with a
    workspace of its own) and with a norm weight of another dtype."""
    g = torch.Generator().manual_seed(1)
    H, inter, M = 512, 8224, 24
    x = torch.randn(M, H, generator=g).bfloat16().to(gpu)
    wgu, wd = (torch.randint(-127, 128, s, generator=g).to(torch.int8).to(gpu) for s in ((2 * inter, H), (H, inter)))
    sgu, sd = (torch.rand(n, generator=g).to(gpu) * 1e-3 for n in (2 * inter, H))
    r = x.flip(0).contiguous() if residual else None
    print("  host mlp", flush=True)
    for nw in (torch.ones(H, device=gpu, dtype=torch.bfloat16), torch.ones(H, device=gpu)):
        def fn():
            return ra.int8_mlp(x, nw, wgu, sgu, wd, sd, 1e-6, r)
        a, p = _pairs(fn, monkeypatch)
        assert a.dtype == p.dtype and torch.equal(a, p)
        st = torch.cuda.Stream()
        st.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(st):
            b = fn()
        torch.cuda.current_stream().wait_stream(st)
        assert torch.equal(a, b)
