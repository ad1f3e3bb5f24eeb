"""The 16-byte row kernels (swiglu, weight quantiser, KV decode, RMSNorm) at
the sizes where their chunks end: rows shorter than a chunk, ragged tails,
rows at odd addresses, the widths at which another form takes over."""
import os
import subprocess

import numpy as np
import pytest
import torch

import rotalabs_accel as ra
from oracle import fallback

HALF = [torch.float16, torch.bfloat16]


def test_fp32_quotient_without_a_division(tmp_path):
    src = os.path.join(os.path.dirname(os.path.abspath(__file__)), "division_f32_check.c")
    exe = str(tmp_path / "division_f32_check")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-mfma", "-o", exe, src, "-lm"], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("dt", HALF + [torch.float32])
@pytest.mark.parametrize("n,k", [(5, 3), (5, 8), (7, 9), (3, 300), (6, 511), (9, 513), (5, 1025), (3, 2051),
                                 (5, 4096), (2, 4099), (3, 8200), (2, 16384), (2, 16391)])
def test_quantize_widths_bit_exact(gpu, dt, n, k):
    """Codes and scales equal the CPU op sequence bit for bit: random rows, an
    all-zero, a tiny-valued, a tie-valued and a NaN row."""
    g = torch.Generator().manual_seed(n * k)
    w = (torch.randn(n + 4, k, generator=g) * 0.02).to(dt)
    w[n] = 0
    w[n + 1] *= 1e-5 if dt == torch.float16 else 1e-33
    w[n + 2] = ((torch.arange(k) % 254 - 127).float() + 0.5).clamp(-127, 127) / 8
    w[n + 2, 0] = 127 / 8
    w[n + 3, k // 2] = float("nan")
    print(f"  quantize {dt} [{n + 4}, {k}]", flush=True)
    # a view one row into a buffer of odd row length: rows at any address
    buf = torch.empty(n + 5, k, dtype=dt, device=gpu)
    buf[1:] = w.to(gpu)
    q, s = ra.quantize_weight_per_channel(buf[1:])
    q_c, s_c = ra.quantize_weight_per_channel(w)
    assert torch.equal(q.cpu(), q_c)
    torch.testing.assert_close(s.cpu(), s_c, rtol=0, atol=0, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", HALF + [torch.float32])
@pytest.mark.parametrize("rows,hidden", [(1, 1), (3, 5), (7, 8), (5, 333), (9, 4104), (300, 2049)])
@pytest.mark.parametrize("bias", [None, "same", torch.float32, torch.float16])
def test_swiglu_tails(gpu, dt, rows, hidden, bias):
    """Chunks that end past n or cross rows, bias chunks in the row or not,
    inputs at an address of no alignment: one output rounding from float64."""
    from rotalabs_accel.kernels.swiglu import swiglu_with_bias
    g = torch.Generator().manual_seed(rows * hidden)
    n = rows * hidden
    flat = [(torch.randn(n + 1, generator=g) * 3).to(dt) for _ in range(2)]
    gate, up = (f.to(gpu)[1:].view(rows, hidden) for f in flat)
    g64, u64 = (f[1:].view(rows, hidden).double().numpy() for f in flat)
    print(f"  swiglu {dt} [{rows}, {hidden}] bias={bias}", flush=True)
    if bias is None:
        y = ra.swiglu_fused(gate, up)
    else:
        bdt = dt if bias == "same" else bias
        bg, bu = (torch.randn(hidden, generator=g).to(bdt) for _ in range(2))
        y = swiglu_with_bias(gate, up, bg.to(gpu), bu.to(gpu))
        g64, u64 = g64 + bg.double().numpy(), u64 + bu.double().numpy()
    ref = fallback.swiglu_f64(g64, u64)
    # the fp32 sums g + b, u + b round once each (2^-24 of them), silu amplifies
    # a relative error of g by at most 1 + |g|; then one rounding to dt
    unit = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -22}[dt]
    np.testing.assert_allclose(y.cpu().double().numpy(), ref, rtol=unit * 1.01 + 2.0 ** -19, atol=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", HALF + [torch.float32])
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (1, 8), (5, 36), (131, 80), (1030, 128), (7, 1000), (2, 8200)])
def test_kv_decode_bit_exact(gpu, dt, rows, cols):
    from rotalabs_accel.speculative import QuantizedTensor
    g = torch.Generator().manual_seed(rows + cols)
    t = (torch.randn(rows, cols, generator=g) * 4).to(dt)
    print(f"  kv decode {dt} [{rows}, {cols}]", flush=True)
    qt = QuantizedTensor(t.to(gpu))
    torch.testing.assert_close(qt.dequantize().cpu(), qt.data.cpu().to(dt) * qt.scale.cpu(), rtol=0, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", HALF)
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("rows,hidden", [(3, 7), (5, 8), (9, 9), (4, 2047), (3, 2056), (5, 4097), (2, 8199), (2, 16383)])
def test_rmsnorm_odd_rows(gpu, dt, wide, rows, hidden):
    """Ragged rows and fp32 weights: bit for bit the exactly rounded
    restatement (its value before the weight, times the weight, for fp32)."""
    g = torch.Generator().manual_seed(rows * hidden)
    x = (torch.randn(rows, hidden, generator=g) * 2).to(dt)
    r = (torch.randn(rows, hidden, generator=g) * 2).to(dt)
    w = (1 + 0.01 * torch.randn(hidden, generator=g)).to(torch.float32 if wide else dt)
    print(f"  rmsnorm {dt} [{rows}, {hidden}] wide={wide}", flush=True)
    name = "f16" if dt == torch.float16 else "bf16"
    for res in (None, r):
        v = x if res is None else x + res
        if res is None:
            y = ra.rmsnorm(x.to(gpu), w.to(gpu), 1e-6).cpu()
        else:
            y = ra.rmsnorm_residual_fused(x.to(gpu), res.to(gpu), w.to(gpu), 1e-6).cpu()
        one = np.ones(hidden, dtype=np.float32)
        n = fallback.rmsnorm_exact_ref(v.float().numpy(), one, 1e-6, name)
        ref = (torch.from_numpy(n) * w.float()).to(w.dtype)
        assert y.dtype == w.dtype and torch.equal(y, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", HALF + [torch.float32])
@pytest.mark.parametrize("rows,hidden", [(1, 1), (3, 5), (7, 8), (5, 333), (6, 4104), (300, 2049), (0, 16)])
def test_swiglu_halves_same_bits(gpu, dt, rows, hidden):
    """The halves read in place give what their contiguous copies give."""
    from rotalabs_accel.kernels.mlp import _swiglu_halves
    g = torch.Generator().manual_seed(hidden)
    gu = (torch.randn(rows, 2 * hidden, generator=g) * 3).to(dt).to(gpu)
    print(f"  swiglu halves {dt} [{rows}, {hidden}]", flush=True)
    ref = ra.swiglu_fused(gu[:, :hidden].contiguous(), gu[:, hidden:].contiguous())
    assert torch.equal(_swiglu_halves(gu), ref)
