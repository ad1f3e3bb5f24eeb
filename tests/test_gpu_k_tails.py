"""The direct-to-LDS and small-batch GEMM kernels at K that are no multiples
of their K tiles (64 and 128): the last tile starts earlier and drops what the
tile before it covered."""
import pytest
import torch

from rotalabs_accel import _backend
from rotalabs_accel.kernels import gemm as gm

pytestmark = pytest.mark.gpu


def _case(M, K, N, dt, gpu):
    """Data whose sums are exact in fp32 and in dt; x rows are followed by NaN."""
    g = torch.Generator().manual_seed(M * K + N)
    x = torch.randint(-1, 2, (M, K), generator=g).float() * (torch.rand(M, K, generator=g) < min(1.0, 127.0 / K))
    q = torch.randint(-1, 2, (N, K), generator=g).to(torch.int8)
    s = torch.full((N,), 2.0 ** -4)
    exact = (x.double() @ q.double().T) * 2.0 ** -4
    xb = torch.full((M, K + 16), float("nan"), dtype=dt, device=gpu)
    xb[:, :K] = x.to(dt)
    return xb[:, :K], q.to(gpu), s.to(gpu), exact.to(gpu)


# Small-batch and split-K: K = 128 + 32 .. 128 + 96 in one or two stages, a
# tail alone in the last split or wave slice; one to four activation tiles and
# the extra-row forms (17, 33).
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("variant", [_backend.VARIANT_BATCH, _backend.VARIANT_SPLITK, _backend.VARIANT_SPLITK_SPREAD])
@pytest.mark.parametrize("M,K,N", [(2, 160, 40), (4, 11040, 300), (16, 224, 1000), (17, 16480, 200), (20, 4192, 515),
                                   (33, 5152, 700), (40, 192, 77), (48, 2144, 260), (64, 11104, 130)])
def test_small_batch_k_tails(gpu, dt, variant, M, K, N):
    x, q, s, exact = _case(M, K, N, dt, gpu)
    print(f"  k tail variant {variant} {dt} M={M} K={K} N={N}", flush=True)
    for _ in range(2):  # the second call finds the counters the first left
        assert torch.equal(gm._int8_gemm_hip(x, q, s, None, variant=variant).double(), exact)


# Tiles: 64 rows (33..64), split plans (65..384), two workgroups per CU (64 and
# 128 rows), the large tiles (the last three); tails of 16, 32 and 48 k, alone
# (K < 128) and after full tiles.
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", [(33, 80, 100), (64, 2096, 8200), (64, 112, 70), (65, 11056, 300), (200, 1072, 1030),
                                   (300, 96, 333), (700, 368, 600), (2000, 304, 520), (1100, 144, 2100),
                                   (2100, 144, 4200), (1300, 80, 6000), (520, 112, 9000)])
def test_tiled_k_tails(gpu, dt, M, K, N):
    x, q, s, exact = _case(M, K, N, dt, gpu)
    print(f"  k tail tiles {dt} M={M} K={K} N={N}", flush=True)
    assert torch.equal(gm._int8_gemm_hip(x, q, s, None, variant=_backend.VARIANT_TILED).double(), exact)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,inter", [(70, 80, 100), (300, 1072, 520), (600, 368, 1000), (128, 64, 17000),
                                       (500, 128, 2050), (600, 368, 5000)])
def test_gateup_tiled_k_tails(gpu, dt, M, K, inter):
    """The gate/up tiles (64 and 128 rows, two workgroups per CU, and the large
    ones): the same sums as the GEMM's, one SwiGLU on top."""
    from rotalabs_accel.kernels.mlp import int8_gateup_swiglu
    x, q, s, exact = _case(M, K, 2 * inter, dt, gpu)
    print(f"  k tail gate/up {dt} M={M} K={K} I={inter}", flush=True)
    a, u = exact[:, :inter], exact[:, inter:]
    ref = (a / (1 + torch.exp(-a))).to(dt).double() * u
    # silu rounded to dt, then the product: an fp32 exp may flip the first rounding
    unit = 2.0 ** -10 if dt == torch.float16 else 2.0 ** -7
    torch.testing.assert_close(int8_gateup_swiglu(x, q, s).double(), ref, rtol=2 * unit, atol=1e-6)
