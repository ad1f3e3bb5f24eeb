// Row-wise and elementwise kernels on the decoder-MLP path:
//  * RMSNorm (the prologue of the gate/up projection),
//  * standalone SwiGLU (the fused path folds it into the gate/up epilogue),
//  * per-output-channel int8 weight quantisation, bit-exact with the CPU.
// All are HBM-bound row/byte work: one workgroup per row, coalesced loads,
// wave64 shuffles + LDS for the row reduction, fp32 math.
#include "ra_common.h"
#include "ra_internal.h"

namespace ra {

constexpr int kRowThreads = 256;

// Workgroup sum, or NaN-propagating maximum (as torch's amax).
template <bool IsMax>
__device__ __forceinline__ float block_reduce(float v, float *smem) {
  v = IsMax ? wave_maximum(v) : wave_sum(v);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) smem[wid] = v;
  __syncthreads();
  float r = smem[0];
#pragma unroll
  for (int i = 1; i < kRowThreads / 64; ++i) r = IsMax ? nan_max(r, smem[i]) : r + smem[i];
  return r;
}

// Workgroup sum of fp64 values (fixed order).
__device__ __forceinline__ double block_sum_f64(double v, double *smem) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) smem[wid] = v;
  __syncthreads();
  double r = smem[0];
#pragma unroll
  for (int i = 1; i < kRowThreads / 64; ++i) r += smem[i];
  return r;
}

// 8 16-bit (or 4 fp32) values of a 16-byte chunk as fp32, and back.
template <int DT>
struct Chunk {
  static constexpr int E = DT == RA_F32 ? 4 : 8;
  static constexpr int SZ = 16 / E;
  static __device__ __forceinline__ float get(const uint4 &v, int e) {
    if constexpr (DT == RA_F32) return reinterpret_cast<const float *>(&v)[e];
    else return Act<DT>::in(reinterpret_cast<const uint16_t *>(&v)[e]);
  }
  static __device__ __forceinline__ void set(uint4 &v, int e, float f) {
    if constexpr (DT == RA_F32) reinterpret_cast<float *>(&v)[e] = f;
    else reinterpret_cast<uint16_t *>(&v)[e] = Act<DT>::out(f);
  }
};

// y = round_y( round_x(v * rsqrt(mean(v^2) + eps)) * w ) with v = x, as
// rmsnorm_torch (src/rotalabs_accel/kernels/normalization.py:43-45): the
// normalised value is stored in x's dtype, then multiplied by the weight in
// the promoted dtype. With a residual r, v = round_s(x + r) in s, the
// promotion of x's and r's dtypes, as rmsnorm_residual_torch (:60-62)
// computes (x + residual) before .float().
// The fp32 squares (exact for 16-bit v) are summed in fp64 and the sum is
// rounded once to fp32: the exactly rounded fp32 sum, whatever the order
// (the reference's fp32 reduction depends on its order; an order-dependent
// last bit of the sum moves rsqrt by an ulp and can flip the 16-bit
// rounding of an element of the row). mean = sum / hidden, + eps and
// rsqrt = 1 / sqrt are fp32 operations, each correctly rounded.
__global__ __launch_bounds__(kRowThreads) void rmsnorm_kernel(const void *__restrict__ x, int64_t ldx,
                                                              int x_dt, const void *__restrict__ r,
                                                              int64_t ldr, int r_dt, int s_dt,
                                                              const void *__restrict__ w,
                                                              int w_dt, void *__restrict__ y,
                                                              int64_t ldy, int y_dt, int hidden,
                                                              float eps) {
  __shared__ double smem[kRowThreads / 64];
  const int64_t row = blockIdx.x;
  auto in = [&](int i) -> float {
    const float v = load_as_f32(x, row * ldx + i, x_dt);
    return r ? round_through(v + load_as_f32(r, row * ldr + i, r_dt), s_dt) : v;
  };
  double ss = 0.0;
  for (int i = threadIdx.x; i < hidden; i += kRowThreads) {
    const float v = in(i);
    ss += (double)fp32_rounded(v * v);
  }
  const float total = (float)block_sum_f64(ss, smem);
  const float rr = 1.0f / sqrtf(total / (float)hidden + eps);
  for (int i = threadIdx.x; i < hidden; i += kRowThreads) {
    const float v = round_through(in(i) * rr, x_dt);
    store_from_f32(y, row * ldy + i, y_dt, v * load_as_f32(w, i, w_dt));
  }
}

// Same arithmetic for x (and r) of one 16-bit dtype, w of that dtype or fp32
// (y: w's) and at least 8 values per row: every thread loads its VPT 16-byte
// chunks of the row (and of r and w) at once, keeps them in registers for the
// normalisation, and stores 16-byte chunks -- one pass over memory with all
// loads in flight, instead of the latency-bound loop above (2-byte accesses,
// x and r read twice). ODD: hidden is no multiple of 8; the last chunk starts
// at hidden - 8, and its values that the chunk before holds too are left out
// of the sum (and stored twice, the same). M=4096 H=4096 bf16 with a
// residual, loop -> this: fp32 weight 67.6 -> 21.9 us, H=4097 67.6 -> 23.4 us.
template <int DT, int WDT, int VPT, bool RES, bool ODD>
__global__ __launch_bounds__(kRowThreads) void rmsnorm_vec_kernel(const uint16_t *__restrict__ x, int64_t ldx,
                                                                  const uint16_t *__restrict__ r, int64_t ldr,
                                                                  const void *__restrict__ w, void *__restrict__ y,
                                                                  int64_t ldy, int hidden, float eps) {
  using A = Act<DT>;
  using W = Chunk<WDT>;
  constexpr int WC = 8 / W::E;  // 16-byte chunks of w and y per chunk of x
  __shared__ double smem[kRowThreads / 64];
  const int64_t row = blockIdx.x;
  const int nch = (hidden + 7) / 8;
  const uint16_t *xr = x + row * ldx;
  const char *wp = static_cast<const char *>(w);
  char *yr = static_cast<char *>(y) + row * ldy * W::SZ;
  auto first = [&](int c) { return ODD ? min(8 * c, hidden - 8) : 8 * c; };
  uint4 xv[VPT], rv[VPT], wv[VPT][WC];
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int i = first(min((int)threadIdx.x + kRowThreads * j, nch - 1));  // clamped: loads stay unconditional
    xv[j] = load16_any(xr + i);
    if (RES) rv[j] = load16_any(r + row * ldr + i);
#pragma unroll
    for (int k = 0; k < WC; ++k) wv[j][k] = load16_any(wp + (int64_t)i * W::SZ + 16 * k);
  }
  // v = x (+ r, rounded to the dtype)
  float v[VPT][8];
  double ss = 0.0;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const uint16_t *h = reinterpret_cast<const uint16_t *>(&xv[j]);
    const uint16_t *hr = reinterpret_cast<const uint16_t *>(&rv[j]);
    const int c = (int)threadIdx.x + kRowThreads * j;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[j][e] = RES ? A::rnd(A::in(h[e]) + A::in(hr[e])) : A::in(h[e]);
      const bool live = c < nch && (!ODD || first(c) + e >= 8 * c);
      if (live) ss += (double)(v[j][e] * v[j][e]);  // exact: 16-bit values square exactly in fp32
    }
  }
  const float total = (float)block_sum_f64(ss, smem);
  const float rr = 1.0f / sqrtf(total / (float)hidden + eps);
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int c = (int)threadIdx.x + kRowThreads * j;
    if (c >= nch) continue;
    uint4 o[WC];
    // (fp32_rounded: v * rr is rounded to fp32, then to 16 bits, not at once)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      W::set(o[e / W::E], e % W::E, A::rnd(fp32_rounded(v[j][e] * rr)) * W::get(wv[j][e / W::E], e % W::E));
#pragma unroll
    for (int k = 0; k < WC; ++k) store16_any(yr + (int64_t)first(c) * W::SZ + 16 * k, o[k]);
  }
}

template <int DT, int WDT, bool RES, bool ODD>
static void rmsnorm_vec_launch(const void *x, int64_t ldx, const void *r, int64_t ldr, const void *w, void *y,
                               int64_t ldy, int64_t rows, int hidden, float eps, hipStream_t s) {
  const int nch = (hidden + 7) / 8;
  const uint16_t *xp = static_cast<const uint16_t *>(x), *rp = static_cast<const uint16_t *>(r);
  const dim3 grid((unsigned)rows), block(kRowThreads);
#define RA_RMS(VPT_)                                                                                              \
  if (nch <= VPT_ * kRowThreads) {                                                                                \
    hipLaunchKernelGGL((rmsnorm_vec_kernel<DT, WDT, VPT_, RES, ODD>), grid, block, 0, s, xp, ldx, rp, ldr, w, y, ldy, \
                       hidden, eps);                                                                              \
    return;                                                                                                       \
  }
  RA_RMS(1) RA_RMS(2) RA_RMS(4) RA_RMS(8)
#undef RA_RMS
}

hipError_t rmsnorm_launch(const void *x, int64_t ldx, int x_dt, const void *r, int64_t ldr, int r_dt,
                          const void *w, int w_dt, void *y, int64_t ldy, int y_dt, int64_t rows, int64_t hidden,
                          float eps, hipStream_t s) {
  const bool vec = (x_dt == RA_F16 || x_dt == RA_BF16) && (w_dt == x_dt || w_dt == RA_F32) && y_dt == w_dt &&
                   (!r || r_dt == x_dt) && hidden >= 8 && hidden <= 8 * 8 * kRowThreads;
  if (vec) {
#define RA_RMS_GO(DT_, WDT_)                                                                                    \
  if (x_dt == DT_ && w_dt == WDT_) {                                                                            \
    auto go = [&](auto res, auto odd) {                                                                         \
      rmsnorm_vec_launch<DT_, WDT_, decltype(res)::value, decltype(odd)::value>(x, ldx, r, ldr, w, y, ldy, rows, \
                                                                                (int)hidden, eps, s);           \
    };                                                                                                          \
    if (r && hidden % 8) go(std::true_type{}, std::true_type{});                                                \
    else if (r) go(std::true_type{}, std::false_type{});                                                        \
    else if (hidden % 8) go(std::false_type{}, std::true_type{});                                               \
    else go(std::false_type{}, std::false_type{});                                                              \
    return hipGetLastError();                                                                                   \
  }
    RA_RMS_GO(RA_F16, RA_F16)
    RA_RMS_GO(RA_F16, RA_F32)
    RA_RMS_GO(RA_BF16, RA_BF16)
    RA_RMS_GO(RA_BF16, RA_F32)
#undef RA_RMS_GO
  }
  const int s_dt = !r ? x_dt : (x_dt == r_dt ? x_dt : RA_F32);  // dtype of x + r
  hipLaunchKernelGGL(rmsnorm_kernel, dim3((unsigned)rows), dim3(kRowThreads), 0, s, x, ldx, x_dt, r, ldr, r_dt,
                     s_dt, w, w_dt, y, ldy, y_dt, (int)hidden, eps);
  return hipGetLastError();
}

// out = silu(g) * u = g / (1 + exp(-g)) * u in fp32, one rounding
// (the Triton kernel's arithmetic, src/rotalabs_accel/kernels/activations.py:69-80).
// (fp32_rounded: the product is rounded to fp32, then to 16 bits, in every form.)
__device__ __forceinline__ float silu_mul(float g, float u) { return fp32_rounded(g / (1.0f + expf(-g)) * u); }

// Bound by HBM (two values read, one written per element). One 16-byte chunk
// of gate and of up per lane: 2-byte accesses moved a quarter of what the
// address units can per instruction (M=4096 I=11008 bf16: 132.9 -> 51.8 us).
// BIAS: 0 none; 2 biases of the same dtype with hidden a whole number of
// chunks (a chunk stays within its row: one bias chunk each); 1 any other.
constexpr int64_t kSwigluMaxBlocks = 1 << 20;  // workgroups per launch (more chunks: each takes several)

template <int DT, int BIAS>
__global__ __launch_bounds__(256) void swiglu_kernel(const void *__restrict__ g, const void *__restrict__ u,
                                                     const void *__restrict__ bg, const void *__restrict__ bu,
                                                     int b_dt, void *__restrict__ o, int64_t n, int64_t hidden) {
  using C = Chunk<DT>;
  const int64_t step = (int64_t)gridDim.x * 256 * C::E;
  for (int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * C::E; i0 < n; i0 += step) {
    int64_t col = BIAS ? (n <= INT32_MAX ? (int64_t)((uint32_t)i0 % (uint32_t)hidden) : i0 % hidden) : 0;
    auto one = [&](float gv, float uv) {
      if (BIAS == 1) {
        gv += load_as_f32(bg, col, b_dt);
        uv += load_as_f32(bu, col, b_dt);
        if (++col == hidden) col = 0;
      }
      return silu_mul(gv, uv);
    };
    if (BIAS != 2 && i0 + C::E > n) {
      for (int64_t i = i0; i < n; ++i) store_from_f32(o, i, DT, one(load_as_f32(g, i, DT), load_as_f32(u, i, DT)));
      return;
    }
    const uint4 gc = load16_any(static_cast<const char *>(g) + i0 * C::SZ);
    const uint4 uc = load16_any(static_cast<const char *>(u) + i0 * C::SZ);
    uint4 bgc, buc, oc;
    if (BIAS == 2) {
      bgc = load16_any(static_cast<const char *>(bg) + col * C::SZ);
      buc = load16_any(static_cast<const char *>(bu) + col * C::SZ);
    }
#pragma unroll
    for (int e = 0; e < C::E; ++e) {
      float gv = C::get(gc, e), uv = C::get(uc, e);
      if (BIAS == 2) {
        gv += C::get(bgc, e);
        uv += C::get(buc, e);
      }
      C::set(oc, e, one(gv, uv));
    }
    store16_any(static_cast<char *>(o) + i0 * C::SZ, oc);
  }
}

template <int BIAS>
static hipError_t swiglu_any(const void *g, const void *u, const void *bg, const void *bu, int b_dt, void *o,
                             int64_t n, int64_t hidden, int dt, hipStream_t s) {
  const int64_t per = 256 * (dt == RA_F32 ? 4 : 8);
  const int64_t blocks = std::min((n + per - 1) / per, kSwigluMaxBlocks);
  const dim3 grid((unsigned)blocks), block(256);
  if (dt == RA_F16)
    hipLaunchKernelGGL((swiglu_kernel<RA_F16, BIAS>), grid, block, 0, s, g, u, bg, bu, b_dt, o, n, hidden);
  else if (dt == RA_BF16)
    hipLaunchKernelGGL((swiglu_kernel<RA_BF16, BIAS>), grid, block, 0, s, g, u, bg, bu, b_dt, o, n, hidden);
  else
    hipLaunchKernelGGL((swiglu_kernel<RA_F32, BIAS>), grid, block, 0, s, g, u, bg, bu, b_dt, o, n, hidden);
  return hipGetLastError();
}

// The same over the two halves of [rows, 2 * hidden] (a gate/up product with
// its biases added, gate columns first): the halves are read in place, where
// two copies made them contiguous before (M=2048 I=11008 bf16: 22.1 after 2 x 16.2 us of copies -> 23.2).
// INROW: hidden is a whole number of chunks, so a chunk stays in its row.
template <int DT, bool INROW>
__global__ __launch_bounds__(256) void swiglu_halves_kernel(const void *__restrict__ gu, int64_t ld,
                                                            void *__restrict__ o, int64_t n, int64_t hidden) {
  using C = Chunk<DT>;
  const int64_t step = (int64_t)gridDim.x * 256 * C::E;
  for (int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * C::E; i0 < n; i0 += step) {
    int64_t row = n <= INT32_MAX ? (int64_t)((uint32_t)i0 / (uint32_t)hidden) : i0 / hidden;
    int64_t col = i0 - row * hidden;
    if constexpr (INROW) {
      const char *gp = static_cast<const char *>(gu) + (row * ld + col) * C::SZ;
      const uint4 gc = load16_any(gp), uc = load16_any(gp + hidden * C::SZ);
      uint4 oc;
#pragma unroll
      for (int e = 0; e < C::E; ++e) C::set(oc, e, silu_mul(C::get(gc, e), C::get(uc, e)));
      store16_any(static_cast<char *>(o) + i0 * C::SZ, oc);
    } else {
      for (int64_t i = i0; i < i0 + C::E && i < n; ++i) {
        store_from_f32(o, i, DT, silu_mul(load_as_f32(gu, row * ld + col, DT), load_as_f32(gu, row * ld + hidden + col, DT)));
        if (++col == hidden) col = 0, ++row;
      }
    }
  }
}

hipError_t swiglu_halves_launch(const void *gu, int64_t ld, void *o, int64_t rows, int64_t hidden, int dt,
                                hipStream_t s) {
  const int64_t n = rows * hidden, per = 256 * (dt == RA_F32 ? 4 : 8);
  const dim3 grid((unsigned)std::min((n + per - 1) / per, kSwigluMaxBlocks)), block(256);
#define RA_HALVES(DT_)                                                                                     \
  if (dt == DT_) {                                                                                         \
    if (hidden % Chunk<DT_>::E == 0)                                                                       \
      hipLaunchKernelGGL((swiglu_halves_kernel<DT_, true>), grid, block, 0, s, gu, ld, o, n, hidden);      \
    else                                                                                                   \
      hipLaunchKernelGGL((swiglu_halves_kernel<DT_, false>), grid, block, 0, s, gu, ld, o, n, hidden);     \
  }
  RA_HALVES(RA_F16) RA_HALVES(RA_BF16) RA_HALVES(RA_F32)
#undef RA_HALVES
  return hipGetLastError();
}

hipError_t swiglu_launch(const void *g, const void *u, void *o, int64_t n, int dt, hipStream_t s) {
  return swiglu_any<0>(g, u, nullptr, nullptr, RA_F32, o, n, n, dt, s);
}

// out = silu(g + bg) * (u + bu) in fp32, one rounding, bias index i % hidden
// (the arithmetic of swiglu_with_bias's Triton kernel,
// src/rotalabs_accel/kernels/swiglu.py:201-218).
hipError_t swiglu_bias_launch(const void *g, const void *u, const void *bg, const void *bu, int b_dt, void *o,
                              int64_t n, int64_t hidden, int dt, hipStream_t s) {
  if (b_dt == dt && hidden % (dt == RA_F32 ? 4 : 8) == 0) return swiglu_any<2>(g, u, bg, bu, b_dt, o, n, hidden, dt, s);
  return swiglu_any<1>(g, u, bg, bu, b_dt, o, n, hidden, dt, s);
}

// Per-row symmetric quantisation, the op sequence of quantize_symmetric(dim=1)
// (src/rotalabs_accel/quantization/symmetric.py:66-80) on the CPU:
//   s = round_w(amax / 127)   IEEE division (built without fast-math)
//   s = 1 if s == 0
//   q = int8(clamp(rint(round_w(w / s)), -128, 127))   rint: half to even
// round_w is the rounding to the weight dtype (identity for fp32). amax
// propagates NaN (torch's amax) and a NaN quotient converts to 0, as the CPU
// conversion does.
__global__ __launch_bounds__(kRowThreads) void quantize_kernel(const void *__restrict__ w, int64_t ldw,
                                                               int w_dt, int K, int8_t *__restrict__ q,
                                                               int64_t ldq, float *__restrict__ scale) {
  __shared__ float smem[kRowThreads / 64];
  const int64_t row = blockIdx.x;
  float amax = 0.f;
  for (int i = threadIdx.x; i < K; i += kRowThreads)
    amax = nan_max(amax, fabsf(load_as_f32(w, row * ldw + i, w_dt)));
  amax = block_reduce<true>(amax, smem);
  float s = round_through(amax / 127.0f, w_dt);
  if (s == 0.0f) s = 1.0f;
  for (int i = threadIdx.x; i < K; i += kRowThreads) {
    const float v = rintf(round_through(load_as_f32(w, row * ldw + i, w_dt) / s, w_dt));
    q[row * ldq + i] = v != v ? (int8_t)0 : (int8_t)(int)fminf(fmaxf(v, -128.0f), 127.0f);
  }
  if (threadIdx.x == 0) scale[row] = s;
}

// Same arithmetic with the row held in registers: one pass over memory, every
// load of the row in flight at once, 16-byte loads and 8-byte (fp32: 4-byte)
// stores at any alignment. WPR waves per row, each lane VPT chunks; the row's
// last chunk starts at K - E where K is no multiple of E (its first values
// are quantised twice, to the same bytes). The kernel above reads the row
// twice in 2-byte accesses and divides each element (N=11008 K=4096 fp16:
// 74.6 -> 25.6 us, HBM-bound).
// The quotient without a division per element: for 16-bit x and scale,
// Markstein's correction as in the KV codec below (same check); for fp32 two
// corrections (the first makes the quotient faithful, the second rounds it
// correctly: rinv is the correctly rounded reciprocal and every residual is
// exact). A tiny, zero-replaced, infinite or NaN scale takes the division.
template <int DT, int VPT, int WPR>
__global__ __launch_bounds__(256) void quantize_vec_kernel(const void *__restrict__ w, int64_t ldw, int N, int K,
                                                           int8_t *__restrict__ q, int64_t ldq,
                                                           float *__restrict__ scale) {
  using C = Chunk<DT>;
  constexpr int T = 64 * WPR;
  __shared__ float smem[kRowThreads / 64];
  const int64_t row = (int64_t)blockIdx.x * (4 / WPR) + (WPR == 4 ? 0 : (int)threadIdx.x / T);
  if (row >= N) return;  // WPR = 1: whole waves, no barrier below; WPR = 4: never
  const int t = threadIdx.x % T;
  const char *wr = static_cast<const char *>(w) + row * ldw * C::SZ;
  const int nch = (K + C::E - 1) / C::E;
  uint4 v[VPT];
  int at[VPT];
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    at[j] = min(C::E * min(t + T * j, nch - 1), K - C::E);  // clamped: loads stay unconditional
    v[j] = load_stream16_any(wr + (int64_t)at[j] * C::SZ);
  }
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j)
#pragma unroll
    for (int e = 0; e < C::E; ++e) amax = nan_max(amax, fabsf(C::get(v[j], e)));
  amax = WPR == 1 ? wave_maximum(amax) : block_reduce<true>(amax, smem);
  float s = round_through(amax / 127.0f, DT);
  if (s == 0.0f) s = 1.0f;
  const float rinv = 1.0f / s;
  const bool fast = s >= (DT == RA_F32 ? 0x1p-90f : 1e-8f) && __builtin_isfinite(s);  // uniform over the row
  int8_t *qr = q + row * ldq;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (t + T * j >= nch) continue;
    uint32_t o[2] = {0, 0};
    if (fast) {
      // every element is finite, so the rounded quotients plus 128 lie in [0, 255]
#pragma unroll
      for (int e = 0; e < C::E; ++e) {
        const float x = C::get(v[j], e);
        const float q0 = x * rinv;
        float q1 = __builtin_fmaf(__builtin_fmaf(-q0, s, x), rinv, q0);
        if constexpr (DT == RA_F32) q1 = __builtin_fmaf(__builtin_fmaf(-q1, s, x), rinv, q1);
        else q1 = Act<DT>::rnd(fp32_rounded(q1));
        const float r = rintf(fp32_rounded(q1));
        o[e / 4] = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_amdgcn_fmed3f(r, -128.0f, 127.0f) + 128.0f, e % 4, o[e / 4]);
      }
      o[0] ^= 0x80808080u;
      o[1] ^= 0x80808080u;
    } else {
#pragma unroll
      for (int e = 0; e < C::E; ++e) {
        const float r = rintf(round_through(fp32_rounded(C::get(v[j], e) / s), DT));
        const int qi = r != r ? 0 : (int)fminf(fmaxf(r, -128.0f), 127.0f);
        o[e / 4] |= (uint32_t)(uint8_t)(int8_t)qi << (8 * (e % 4));
      }
    }
    if constexpr (C::E == 8) store8_any(qr + at[j], o[0], o[1]);
    else *reinterpret_cast<u32_any *>(qr + at[j]) = o[0];
  }
  if (t == 0) scale[row] = s;
}

// One wave per row up to 8 chunks per lane (K <= 4096 in 16 bits, 2048 in
// fp32), four waves up to 32 chunks per wave (16384 / 8192); longer rows and
// rows shorter than a chunk take the loop kernel.
template <int DT>
static bool quantize_vec_launch(const void *w, int64_t ldw, int64_t N, int64_t K, int8_t *q, int64_t ldq,
                                float *scale, hipStream_t s) {
  constexpr int E = Chunk<DT>::E;
  if (K < E) return false;
  const int64_t nch = (K + E - 1) / E;
#define RA_QVEC(VPT_, WPR_)                                                                                        \
  if (nch <= 64 * WPR_ * VPT_) {                                                                                   \
    hipLaunchKernelGGL((quantize_vec_kernel<DT, VPT_, WPR_>), dim3((unsigned)((N + 4 / WPR_ - 1) / (4 / WPR_))),   \
                       dim3(256), 0, s, w, ldw, (int)N, (int)K, q, ldq, scale);                                    \
    return true;                                                                                                   \
  }
  RA_QVEC(1, 1) RA_QVEC(2, 1) RA_QVEC(4, 1) RA_QVEC(8, 1) RA_QVEC(4, 4) RA_QVEC(8, 4)
#undef RA_QVEC
  return false;
}

hipError_t quantize_launch(const void *w, int64_t ldw, int w_dt, int64_t N, int64_t K, int8_t *q,
                           int64_t ldq, float *scale, hipStream_t s) {
  if (w_dt == RA_F16 ? quantize_vec_launch<RA_F16>(w, ldw, N, K, q, ldq, scale, s)
      : w_dt == RA_BF16 ? quantize_vec_launch<RA_BF16>(w, ldw, N, K, q, ldq, scale, s)
                        : quantize_vec_launch<RA_F32>(w, ldw, N, K, q, ldq, scale, s))
    return hipGetLastError();
  hipLaunchKernelGGL(quantize_kernel, dim3((unsigned)N), dim3(kRowThreads), 0, s, w, ldw, w_dt, (int)K, q,
                     ldq, scale);
  return hipGetLastError();
}

// Per-row symmetric quantisation of a KV-cache tensor, as QuantizedTensor
// (src/rotalabs_accel/speculative/kv_compression.py:51-78, per_channel) on
// the CPU, with every intermediate in the tensor's dtype t:
//   s = round_t(max(round_t(amax / qmax), 1e-8))      qmax = 2^(bits-1) - 1
//   q = int8(clamp(rint(round_t(x / s)), -qmax-1, qmax)), NaN -> 0
// (fp16 rounds the 1e-8 floor to 0, so an all-zero row gives 0/0 = NaN, which
// the CPU's float -> int8 conversion turns into 0). The scale is stored in t.
__global__ __launch_bounds__(kRowThreads) void quantize_rows_kernel(const void *__restrict__ t, int64_t ldt,
                                                                    int t_dt, int cols, int qmax,
                                                                    int8_t *__restrict__ q, int64_t ldq,
                                                                    void *__restrict__ scale) {
  __shared__ float smem[kRowThreads / 64];
  const int64_t row = blockIdx.x;
  float amax = 0.f;
  for (int i = threadIdx.x; i < cols; i += kRowThreads)
    amax = nan_max(amax, fabsf(load_as_f32(t, row * ldt + i, t_dt)));
  amax = block_reduce<true>(amax, smem);
  const float s = round_through(nan_max(round_through(amax / (float)qmax, t_dt), 1e-8f), t_dt);
  for (int i = threadIdx.x; i < cols; i += kRowThreads) {
    const float v = round_through(load_as_f32(t, row * ldt + i, t_dt) / s, t_dt);
    const float r = rintf(v);
    q[row * ldq + i] = r != r ? (int8_t)0 : (int8_t)(int)fminf(fmaxf(r, (float)(-qmax - 1)), (float)qmax);
  }
  if (threadIdx.x == 0) store_from_f32(scale, row, t_dt, s);
}

// Same arithmetic for short 16-bit rows (cols % 8 == 0, cols <= 512, 16-byte
// aligned rows; e.g. head_dim-wide KV rows): L = cols / 8 lanes per row
// (rounded up to a power of two), 64 / L rows per wave, each lane one 16-byte
// chunk of 8 values (4 rows' chunks loaded at once), the row maximum by lane
// shuffles within the group, 8-byte stores of the 8 quantised values -- no
// per-row workgroup.
template <int DT, int L>
__global__ __launch_bounds__(256) void quantize_rows_short_kernel(const uint16_t *__restrict__ t, int64_t ldt,
                                                                  int64_t rows, int cols, int qmax,
                                                                  int8_t *__restrict__ q, int64_t ldq,
                                                                  uint16_t *__restrict__ scale) {
  using A = Act<DT>;
  constexpr int U = 4;                       // rows per lane group, loads in flight together
  constexpr int RPW = 64 / L;                // rows per wave and pass
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int c = lane % L;                    // 16-byte chunk of this lane
  const int64_t row0 = ((int64_t)blockIdx.x * 4 + wid) * (RPW * U) + lane / L;
  const int cc = 8 * c < cols ? c : 0;       // clamped: loads stay unconditional
  const float qf = (float)qmax, rq = 1.0f / qf, qlo = -qf - 1.0f, qhi = qf;
  uint4 v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int64_t rr = row0 + (int64_t)u * RPW;
    rr = rr < rows ? rr : rows - 1;
    v[u] = load_stream16(t + rr * ldt + 8 * cc);  // read once: non-temporal (72 -> 66 us on 256 MiB)
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t row = row0 + (int64_t)u * RPW;
    const bool live = row < rows && 8 * c < cols;
    const uint16_t *h = reinterpret_cast<const uint16_t *>(&v[u]);
    float x[8], amax = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = A::in(h[e]);
      amax = nan_max(amax, fabsf(x[e]));  // NaN propagates, as torch's amax
    }
    if (!live) amax = 0.f;
#pragma unroll
    for (int off = L / 2; off >= 1; off >>= 1) amax = nan_max(amax, __shfl_xor(amax, off, 64));
    // amax / qmax by the same correction (exact for every finite 16-bit amax
    // and qmax = 127 or 7, checked exhaustively; inf and NaN pass through)
    const float d0 = amax * rq;
    const float d = __builtin_isfinite(d0) ? __builtin_fmaf(__builtin_fmaf(-d0, qf, amax), rq, d0) : d0;
    const float sc = A::rnd(nan_max(A::rnd(fp32_rounded(d)), 1e-8f));
    if (!live) continue;
    // x / sc correctly rounded to fp32 without a division per element:
    // Markstein's correction of x * RN(1/sc) by one residual FMA. For every
    // 16-bit x and 16-bit sc >= 1e-8 with |x / sc| <= 256 (the codec's range:
    // |x| <= amax, sc ~ amax / qmax) it rounds to the same 16-bit value as the
    // IEEE quotient (checked exhaustively on the CPU, both formats). A zero
    // scale (fp16 rounds the 1e-8 floor to 0) or an infinite one (a row
    // holding inf) keeps the plain product x * (1 / sc): +-inf / NaN for
    // x / 0, 0 / NaN for x / inf, as the quotient.
    const float rinv = 1.0f / sc;
    uint32_t lo = 0, hi = 0;
    if (sc != 0.0f && __builtin_isfinite(sc)) {
      // Finite, nonzero scale: every element is finite (a NaN or inf element
      // makes amax, hence sc, NaN or inf), so the clamped integers plus 128
      // lie in [0, 255]; convert and pack them four at a time, then flip the
      // sign bits.
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float q0 = x[e] * rinv;
        const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, sc, x[e]), rinv, q0);
        // (the rounded value goes through a register again: otherwise the
        // compiler re-rounds the integral rint result to 16 bits)
        const float r = rintf(fp32_rounded(A::rnd(fp32_rounded(q1))));
        const float b = __builtin_amdgcn_fmed3f(r, qlo, qhi) + 128.0f;
        if (e < 4) lo = __builtin_amdgcn_cvt_pk_u8_f32(b, e, lo);
        else hi = __builtin_amdgcn_cvt_pk_u8_f32(b, e - 4, hi);
      }
      lo ^= 0x80808080u;
      hi ^= 0x80808080u;
    } else {
      // Zero scale (fp16 rounds the 1e-8 floor to 0), infinite or NaN: the
      // plain product x * (1 / sc) is the quotient's +-inf / NaN / 0; NaN
      // converts to 0.
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float r = rintf(A::rnd(fp32_rounded(x[e] * rinv)));
        const int qi = r != r ? 0 : (int)__builtin_amdgcn_fmed3f(r, qlo, qhi);
        const uint32_t b = (uint32_t)(uint8_t)(int8_t)qi;
        if (e < 4) lo |= b << (8 * e);
        else hi |= b << (8 * (e - 4));
      }
    }
    store8(q + row * ldq + 8 * c, lo, hi);
    if (c == 0) scale[row] = A::out(sc);
  }
}

template <int DT>
static void quantize_rows_short_launch(const void *t, int64_t ldt, int64_t rows, int cols, int qmax, int8_t *q,
                                       int64_t ldq, void *scale, hipStream_t s) {
  const uint16_t *tp = static_cast<const uint16_t *>(t);
  uint16_t *sp = static_cast<uint16_t *>(scale);
  const int need = cols / 8;
#define RA_QROWS(L_)                                                                                \
  if (need <= L_) {                                                                                 \
    const int64_t blocks = (rows + 4 * 4 * (64 / L_) - 1) / (4 * 4 * (64 / L_));                  \
    hipLaunchKernelGGL((quantize_rows_short_kernel<DT, L_>), dim3((unsigned)blocks), dim3(256), 0, s, tp, ldt, \
                       rows, cols, qmax, q, ldq, sp);                                               \
    return;                                                                                         \
  }
  RA_QROWS(1) RA_QROWS(2) RA_QROWS(4) RA_QROWS(8) RA_QROWS(16) RA_QROWS(32) RA_QROWS(64)
#undef RA_QROWS
}

hipError_t quantize_rows_launch(const void *t, int64_t ldt, int t_dt, int64_t rows, int64_t cols, int bits,
                                int8_t *q, int64_t ldq, void *scale, hipStream_t s) {
  const int qmax = (1 << (bits - 1)) - 1;
  const bool short_rows = (t_dt == RA_F16 || t_dt == RA_BF16) && cols % 8 == 0 && cols <= 512 && ldt % 8 == 0 &&
                          ldq % 8 == 0 && !(reinterpret_cast<uintptr_t>(t) & 15) &&
                          !(reinterpret_cast<uintptr_t>(q) & 7) && rows * 64 < ((int64_t)1 << 31);
  if (short_rows) {
    if (t_dt == RA_F16) quantize_rows_short_launch<RA_F16>(t, ldt, rows, (int)cols, qmax, q, ldq, scale, s);
    else quantize_rows_short_launch<RA_BF16>(t, ldt, rows, (int)cols, qmax, q, ldq, scale, s);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(quantize_rows_kernel, dim3((unsigned)rows), dim3(kRowThreads), 0, s, t, ldt, t_dt, (int)cols,
                     qmax, q, ldq, scale);
  return hipGetLastError();
}

// The codec's way back: out = round_t(q * s_row), one fp32 product of exact
// factors rounded once, as torch's data.to(t) * scale (every int8 is exact in
// t) -- in one pass where the two torch ops write and re-read the converted
// codes. HBM-bound; kDeqChunks chunks of 8 codes per lane keep 32 bytes of
// loads in flight each (bf16 [8, 32, 4096, 128]: 372.6 us for the two ops ->
// 61.9 us). INROW: whole rows of chunks (cols % 8 == 0).
constexpr int kDeqChunks = 4;
template <int DT, bool INROW>
__global__ __launch_bounds__(256) void dequantize_rows_kernel(const int8_t *__restrict__ q,
                                                              const void *__restrict__ scale,
                                                              void *__restrict__ out, int64_t n, int64_t cols) {
  const int c0 = (int)(blockIdx.x * (256 * kDeqChunks) + threadIdx.x);
  auto value = [&](uint32_t w, int b, float s) { return (float)(int8_t)(w >> (8 * b)) * s; };
  if constexpr (INROW) {
    const uint32_t cpr = (uint32_t)(cols / 8);  // chunks per row
    const int nch = (int)(n / 8);
    uint2 v[kDeqChunks];
    float s[kDeqChunks];
#pragma unroll
    for (int j = 0; j < kDeqChunks; ++j) {
      const int c = min(c0 + 256 * j, nch - 1);  // clamped: loads stay unconditional
      const u32x2_t d = __builtin_nontemporal_load(reinterpret_cast<const u32x2_any *>(q + (int64_t)8 * c));
      v[j] = make_uint2(d.x, d.y);
      s[j] = load_as_f32(scale, (uint32_t)c / cpr, DT);
    }
#pragma unroll
    for (int j = 0; j < kDeqChunks; ++j) {
      const int c = c0 + 256 * j;
      if (c >= nch) continue;
      char *o = static_cast<char *>(out) + (int64_t)8 * c * Chunk<DT>::SZ;
      uint4 r[2];
#pragma unroll
      for (int e = 0; e < 8; ++e)
        Chunk<DT>::set(r[e / Chunk<DT>::E], e % Chunk<DT>::E, value(e < 4 ? v[j].x : v[j].y, e % 4, s[j]));
      store16_any(o, r[0]);
      if (DT == RA_F32) store16_any(o + 16, r[1]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < kDeqChunks; ++j) {
      const int64_t i0 = (int64_t)8 * (c0 + 256 * j);
      int64_t row = i0 / cols, col = i0 - row * cols;
      for (int64_t i = i0; i < i0 + 8 && i < n; ++i) {
        store_from_f32(out, i, DT, (float)q[i] * load_as_f32(scale, row, DT));
        if (++col == cols) col = 0, ++row;
      }
    }
  }
}

// A launch covers whole rows of at most 2^33 values (32-bit chunk indices;
// one row of up to 2^31 - 1 values always fits).
constexpr int64_t kDeqMaxValues = (int64_t)1 << 33;

hipError_t dequantize_rows_launch(const int8_t *q, const void *scale, int t_dt, int64_t rows, int64_t cols, void *out,
                                  hipStream_t s) {
  constexpr int64_t per = 256 * kDeqChunks * 8;
  const size_t sz = t_dt == RA_F32 ? 4 : 2;
  const int64_t step = kDeqMaxValues / cols;
  for (int64_t r = 0; r < rows; r += step) {
    const int64_t n = std::min(step, rows - r) * cols;
    const dim3 grid((unsigned)((n + per - 1) / per)), block(256);
    const int8_t *qr = q + r * cols;
    const void *sr = static_cast<const char *>(scale) + r * sz;
    void *o = static_cast<char *>(out) + r * cols * sz;
#define RA_DEQ_GO(DT_, IN_) \
  hipLaunchKernelGGL((dequantize_rows_kernel<DT_, IN_>), grid, block, 0, s, qr, sr, o, n, cols)
    if (cols % 8 == 0) {
      if (t_dt == RA_F16) RA_DEQ_GO(RA_F16, true);
      else if (t_dt == RA_BF16) RA_DEQ_GO(RA_BF16, true);
      else RA_DEQ_GO(RA_F32, true);
    } else {
      if (t_dt == RA_F16) RA_DEQ_GO(RA_F16, false);
      else if (t_dt == RA_BF16) RA_DEQ_GO(RA_BF16, false);
      else RA_DEQ_GO(RA_F32, false);
    }
#undef RA_DEQ_GO
  }
  return hipGetLastError();
}

}  // namespace ra
