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
