"""The register-staged MFMA GEMM (fp32 activations; rows of any length and
alignment): every tile geometry at sizes where tiles, K tiles and chunks end,
against exact sums, the VALU kernel and float64."""
import pytest
import torch

import rotalabs_accel as ra
from rotalabs_accel import _backend
from rotalabs_accel.kernels import gemm as gm

pytestmark = pytest.mark.gpu
DTYPES = [torch.float16, torch.bfloat16, torch.float32]


def _run(x, q, s, b=None, variant=_backend.VARIANT_STAGED):
    return gm._int8_gemm_hip(x, q, s, b, variant=variant)


# 16-bit geometries: 32 x 32 (the first six), 32 x 64 (77 rows), 64 x 64
# (2 x 129 tiles), 128 x 128 (1032 tiles of 64 x 64); fp32: 32 x 64, and
# 64 x 128 for the last two.
@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("M,K,N", [(1, 16, 1), (5, 17, 33), (33, 63, 64), (2, 127, 1000), (31, 129, 95), (3, 1009, 70),
                                   (77, 1000, 4101), (128, 333, 8200), (512, 71, 8200), (300, 193, 8200)])
def test_exact_sums_any_alignment(gpu, dt, M, K, N):
    """Integer data whose sums are exact in fp32 and in the output type: every
    output is the exact sum. Rows sit at odd addresses with NaN (x) and 127
    (weights) between and behind them: nothing past K may reach a product."""
    g = torch.Generator().manual_seed(M * K + N)
    x = torch.randint(-1, 2, (M, K), generator=g).float() * (torch.rand(M, K, generator=g) < min(1.0, 127.0 / K))
    q = torch.randint(-1, 2, (N, K), generator=g).to(torch.int8)
    s = torch.full((N,), 2.0 ** -4)
    b = torch.randint(-8, 9, (N,), generator=g).float() * 2.0 ** -4
    exact = ((x.double() @ q.double().T) * 2.0 ** -4 + b.double()).to(gpu)
    print(f"  staged exact {dt} M={M} K={K} N={N}", flush=True)
    xb = torch.full((M * (K + 3) + 1,), float("nan"), dtype=dt, device=gpu)
    xv = xb[1:].view(M, K + 3)[:, :K]
    xv.copy_(x.to(dt))
    wb = torch.full((N * (K + 5) + 3,), 127, dtype=torch.int8, device=gpu)
    wv = wb[3:].view(N, K + 5)[:, :K]
    wv.copy_(q)
    lib = _backend.load()
    y = torch.empty(M, N, dtype=dt, device=gpu)
    bias = b.to(dt).to(gpu)
    sc = s.to(gpu)
    code = _backend.dtype_code(dt)
    _backend.check(lib.ra_w8a16_gemm_ex(xv.data_ptr(), K + 3, code, wv.data_ptr(), K + 5, sc.data_ptr(),
                                        bias.data_ptr(), code, y.data_ptr(), N, M, N, K, _backend.VARIANT_STAGED, None,
                                        0, _backend.stream_handle(gpu)))
    assert torch.equal(y.double(), exact)


@pytest.mark.parametrize("M,K,N", [(3, 300, 400), (64, 1000, 300), (200, 4096, 512), (512, 2048, 4096)])
@pytest.mark.parametrize("spread", [0, 12])
def test_fp32_error_is_no_larger_than_the_valu_kernels(gpu, M, K, N, spread):
    """The error against float64 stays at or below that of the plain fp32 dot
    products. Activations whose magnitudes differ by 2^spread make sums of a
    few large terms, where the order of the additions decides which of the two
    is closer: there the bound is one unit in the last place (2^-23) of the
    norm, about four independent half-unit roundings of the full sum -- a run
    of 8 MFMAs, its fold, the K groups and the scale make fewer than 16."""
    g = torch.Generator().manual_seed(K + spread)
    x = torch.randn(M, K, generator=g) * torch.exp2(torch.rand(M, K, generator=g) * spread)
    q = torch.randint(-127, 128, (N, K), generator=g).to(torch.int8)
    s = torch.rand(N, generator=g) * 1e-3
    x, q, s = x.to(gpu), q.to(gpu), s.to(gpu)
    print(f"  staged fp32 error M={M} K={K} N={N} spread={spread}", flush=True)
    ref = (x.double() @ q.double().T) * s.double()
    err = [((_run(x, q, s, variant=v).double() - ref).norm() / ref.norm()).item()
           for v in (_backend.VARIANT_STAGED, _backend.VARIANT_GENERIC)]
    assert err[0] <= (max(err[1], 2.0 ** -23) if spread else err[1]), err


def test_fp32_infinities_and_nan(gpu):
    """Rows holding an infinity, a NaN (payload in the low bits only), the
    largest and subnormal values: infinite, NaN and finite where the VALU
    kernel's outputs are."""
    g = torch.Generator().manual_seed(3)
    x = torch.randn(40, 200, generator=g)
    x[1, 5] = float("inf")
    x[2, 6] = float("-inf")
    x[3, 7] = torch.tensor(0x7F800001, dtype=torch.int32).view(torch.float32)
    x[4, 8], x[4, 9] = float("inf"), float("-inf")
    x[5] = 3.0e38
    x[6] = 1e-42
    q = torch.randint(1, 128, (70, 200), generator=g).to(torch.int8)
    q[:, 9] = -3
    s = torch.full((70,), 0.5)
    x, q, s = x.to(gpu), q.to(gpu), s.to(gpu)
    print("  staged fp32 special values", flush=True)
    y, ref = _run(x, q, s), _run(x, q, s, variant=_backend.VARIANT_GENERIC)
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
    assert torch.equal(torch.sign(y[y.isinf()]), torch.sign(ref[ref.isinf()]))
    fin = ref.isfinite()
    # Two orders of one fp32 sum: each within its roundings (fewer than 32 on a
    # term's way in either) of the sum of magnitudes. 1e-42: below the smallest
    # normal bf16 the low planes may flush to zero.
    bound = 32 * 2.0 ** -24 * (x.double().abs() @ q.double().abs().T) * s.double() + 1e-36
    assert ((y.double() - ref.double()).abs()[fin] <= bound[fin]).all()


@pytest.mark.parametrize("dt", DTYPES)
def test_selected_where_it_is_ahead(gpu, dt):
    """The automatic choice runs it for unaligned operands and fp32 and the
    module's outputs are its outputs."""
    lib = _backend.load()
    code = _backend.dtype_code(dt)
    assert lib.ra_w8a16_gemm_select(77, 4101, 1000 if dt == torch.float32 else 1001, code) == _backend.VARIANT_STAGED
    assert lib.ra_w8a16_gemm_select(8, 64, 15, code) == _backend.VARIANT_GENERIC
    g = torch.Generator().manual_seed(9)
    x = torch.randn(2, 19, 301, generator=g).to(dt).to(gpu)
    q = torch.randint(-127, 128, (77, 301), generator=g).to(torch.int8).to(gpu)
    s = (torch.rand(77, generator=g) * 1e-2).to(gpu)
    y = ra.int8_gemm(x, q, s)
    assert torch.equal(y, _run(x.reshape(-1, 301), q, s).view(2, 19, 77))
