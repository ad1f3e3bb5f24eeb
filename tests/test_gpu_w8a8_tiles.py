"""The int8 x int8 GEMM's tile configurations: one shape past and one within
each, against exact integer sums."""
import pytest
import torch

from rotalabs_accel.kernels import quantized_matmul as qm

pytestmark = pytest.mark.gpu


# 64 x 64, 64 x 128, 128 x 128, 128 x 192 and the whole-round tiles; K % 128
# == 64: 64 x 128, 128 x 128 and 256 x 128 in 64-k stages; one K tile, rows and
# columns one past a tile.
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", [(17, 128, 70), (65, 256, 8129), (129, 384, 16129), (200, 128, 30000), (257, 256, 24500),
                                   (18, 64, 33), (129, 192, 8200), (300, 320, 11000), (700, 64, 20000)])
@pytest.mark.parametrize("bias", [False, True])
def test_tiles_exact(gpu, dt, M, K, N, bias):
    g = torch.Generator().manual_seed(M + K + N)
    xq = torch.randint(-128, 128, (M, K), generator=g).to(torch.int8)
    w = torch.randint(-128, 128, (N, K), generator=g).to(torch.int8)
    xs = (torch.rand(M, generator=g) * 1e-2).to(dt)
    s = torch.rand(N, generator=g) * 1e-2
    b = torch.randn(N, generator=g) if bias else None
    print(f"  w8a8 tiles {dt} M={M} K={K} N={N} bias={bias}", flush=True)
    y = qm.w8a8_gemm(xq.to(gpu), xs.to(gpu), w.to(gpu), s.to(gpu), None if b is None else b.to(gpu))
    acc = (xq.to(gpu).double() @ w.to(gpu).double().t()).cpu()
    ref = (acc.float() * xs.float()[:, None]) * s[None, :]
    ref = (ref if b is None else ref + b).to(dt)
    assert torch.equal(y.cpu(), ref)
