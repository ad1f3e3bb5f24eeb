// Register-staged W8A16 MFMA GEMM for the operands the direct-to-LDS kernels
// cannot take: fp32 activations, and 16-bit activations or weights whose rows
// start or end anywhere (K % 16 != 0, odd addresses or row strides).
//
// Replaces the reference's Triton tile loop (src/rotalabs_accel/kernels/
// gemm.py:113-138) for those inputs; the VALU kernel (ra_generic.hip), which
// ran them all before, needs two VALU instructions per product. Whole calls,
// before -> after: fp32 M=512 K=N=4096 4217 -> 61.7 us, error against float64
// 1.6e-7 -> 8.8e-8; fp16 M=77 K=1000 N=4101 186.8 -> 13.5 us (8.1 the kernel).
// Bound by the waves' own instructions (splitting x, dequantising, LDS reads),
// not by the MFMAs or memory: fp32 M=32 K=N=4096 takes as long per K tile.
//
//  * fp32 activations: x = hi + mid + lo, three bf16 values cut from the 24
//    bits of x (8 each, truncated, so every residual and the split itself are
//    exact); int8 weights are exact in bf16, so every product of the three
//    planes is exact and the result differs from an fp32 dot product only by
//    the order of its fp32 sums. mid and lo products sum in an accumulator of
//    their own (2^-8 of the result: their roundings do not matter); the hi
//    products' running sum moves into a second accumulator every kFold K
//    tiles, which keeps the rounding chain about as short as that of 64 lanes
//    with a sum each. Infinities and NaN go through the hi plane alone.
//  * Tile (32*BMB*WM) x (32*BNB*WN) x 64, WM x WN waves, each BMB x BNB blocks
//    of v_mfma_f32_32x32x16; KG groups of WM*WN waves share the tile and take
//    a contiguous share of K each (their sums meet in LDS, in group order):
//    where M x N gives few tiles, the groups keep more loads in flight and
//    two or more waves per SIMD.
//  * Global -> registers -> LDS, two K tiles of registers in flight, LDS
//    double-buffered. The loads are 16 bytes at any address. A chunk that
//    would pass K starts at K - its length instead and is shifted into place
//    with zeros behind it: no access leaves the row, and what lies behind a
//    row never meets a product. The fp32 split happens on the way into LDS.
//  * LDS layout, swizzles and the K permutation of the MFMA sub-steps are
//    those of the direct-to-LDS kernel (ra_tiled.hip): activation rows of
//    128 bytes per plane, weight rows of 64 int8, dequantised after the read.
#include "ra_common.h"
#include "ra_internal.h"

namespace ra {
namespace staged {

constexpr int BK = 64;
constexpr int kFold = 2;  // K tiles per chain of the hi products (8 MFMAs), and per turn of the K loop

template <int XDT, int BMB, int BNB, int WM, int WN, int KG>
struct Geo {
  static constexpr int P = XDT == RA_F32 ? 3 : 1;  // activation planes
  static constexpr int BM = 32 * BMB * WM, BN = 32 * BNB * WN;
  static constexpr int TG = 64 * WM * WN;  // threads of a group
  static constexpr int THREADS = TG * KG;
  static constexpr int A_PLANE = BM * 128, B_BYTES = BN * 64;
  static constexpr int STAGE = P * A_PLANE + B_BYTES;
  static constexpr int AC = BM * 8 / TG, BC = BN * 4 / TG;  // chunks per thread and K tile
  static constexpr int LDS = 2 * KG * STAGE;
  static_assert(BM * 8 % TG == 0 && BN * 4 % TG == 0, "chunks must split evenly");
  static_assert(LDS <= 160 * 1024, "LDS");
  static_assert((KG - 1) * BM * BN * 4 <= LDS, "the groups' sums reuse the stages");
};

// v >> (8 * s) over 16 bytes, zeros shifted in (s >= 16: zero).
__device__ __forceinline__ uint4 shr_bytes(uint4 v, int s) {
  uint64_t lo = v.x | (uint64_t)v.y << 32, hi = v.z | (uint64_t)v.w << 32;
  if (s >= 16) lo = hi = 0;
  else if (s >= 8) lo = hi >> (8 * (s - 8)), hi = 0;
  else if (s > 0) lo = lo >> (8 * s) | hi << (64 - 8 * s), hi >>= 8 * s;
  return make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
}

// 8 fp32 values -> three chunks of 8 bf16 (hi, mid, lo).
__device__ __forceinline__ void split8(const uint4 &v0, const uint4 &v1, uint4 (&o)[3]) {
  const uint32_t u[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
  uint32_t *const out[3] = {&o[0].x, &o[1].x, &o[2].x};
  float special = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    float r[2], l[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t b = u[e + k];
      r[k] = __uint_as_float(b) - __uint_as_float(b & 0xffff0000u);
      l[k] = r[k] - __uint_as_float(__float_as_uint(r[k]) & 0xffff0000u);
      special = nan_max(special, l[k]);
    }
    out[0][e / 2] = __builtin_amdgcn_perm(u[e + 1], u[e], 0x07060302u);
    out[1][e / 2] = pack_hi16(r[0], r[1]);
    out[2][e / 2] = pack_hi16(l[0], l[1]);
  }
  if (special != special) {
    // an infinity (inf - inf above) or a NaN: itself in hi (a NaN made quiet,
    // its upper half could be an infinity's), zero in mid and lo
    auto half = [&](uint32_t b, int p) -> uint32_t {
      const float r = __uint_as_float(b) - __uint_as_float(b & 0xffff0000u);
      if ((b & 0x7f800000u) == 0x7f800000u) return p ? 0 : (b & 0x007fffffu ? 0x7fc0u : b >> 16);
      if (p == 0) return b >> 16;
      return __float_as_uint(p == 1 ? r : r - __uint_as_float(__float_as_uint(r) & 0xffff0000u)) >> 16;
    };
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int e = 0; e < 8; e += 2) out[p][e / 2] = half(u[e], p) | half(u[e + 1], p) << 16;
  }
}

template <int XDT, int BMB, int BNB, int WM, int WN, int KG>
__global__ __launch_bounds__(64 * WM * WN * KG) void staged_kernel(
    const void *__restrict__ x, int64_t ldx, const int8_t *__restrict__ w, int64_t ldw,
    const float *__restrict__ scale, const void *__restrict__ bias, int bias_dt, void *__restrict__ y, int64_t ldy,
    int M, int N, int K, int tiles_m, int tiles_n) {
  using G = Geo<XDT, BMB, BNB, WM, WN, KG>;
  using Ac = Act<XDT == RA_F16 ? RA_F16 : RA_BF16>;
  constexpr int P = G::P, AC = G::AC, BC = G::BC;
  constexpr int XSZ = XDT == RA_F32 ? 4 : 2;
  constexpr int AR = XDT == RA_F32 ? 2 : 1;  // 16-byte loads per activation chunk
  __shared__ __attribute__((aligned(1024))) uint8_t lds[G::LDS];

  // ---- tile (XCD-aware: an XCD runs consecutive tiles, M fastest within
  // groups of 8 row tiles, so the row tiles of a weight column share its L2)
  const int T = tiles_m * tiles_n, b = blockIdx.x;
  const int xcd = b & 7, per = T >> 3, rem = T & 7;
  const int t = xcd * per + (xcd < rem ? xcd : rem) + (b >> 3);
  constexpr int GM = 8;
  const int span = GM * tiles_n, first_m = (t / span) * GM, gm = min(tiles_m - first_m, GM);
  const int m0 = (first_m + (t % span) % gm) * G::BM, n0 = (t % span) / gm * G::BN;

  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wid / (WM * WN), wg = wid % (WM * WN);
  const int wm = wg / WN, wn = wg % WN;
  const int tid = threadIdx.x % G::TG;
  uint8_t *const stages = lds + kg * 2 * G::STAGE;

  // K tiles of this group: kt0 .. kt0 + n - 1 (tiles past K are all zeros)
  const int KT = (K + BK - 1) / BK, n = (KT + KG - 1) / KG, kt0 = kg * n;

  // ---- staging: chunk i of a thread is row i * (TG / 8) + tid / 8 (weights:
  // / 4), chunk tid % 8 (% 4). Rows past M / N are clamped, never stored.
  const int ca = tid & 7, cb = tid & 3;
  const char *ap[AC];
  const int8_t *bp[BC];
  int a_dst[AC], b_dst[BC];
#pragma unroll
  for (int i = 0; i < AC; ++i) {
    const int row = i * (G::TG / 8) + (tid >> 3);
    ap[i] = static_cast<const char *>(x) + (int64_t)min(m0 + row, M - 1) * ldx * XSZ;
    a_dst[i] = row * 128 + ((ca ^ ((row >> 1) & 7)) << 4);
  }
#pragma unroll
  for (int i = 0; i < BC; ++i) {
    const int row = i * (G::TG / 4) + (tid >> 2);
    bp[i] = w + (int64_t)min(n0 + row, N - 1) * ldw;
    b_dst[i] = P * G::A_PLANE + row * 64 + ((cb ^ ((row >> 2) & 3)) << 4);
  }
  struct Regs {
    uint4 a[AC][AR], b[BC];
  };
  auto load = [&](Regs &r, int kt) __attribute__((always_inline)) {
    const int k0 = (kt0 + kt) * BK;
#pragma unroll
    for (int q = 0; q < AR; ++q) {
      const int64_t ka = min(k0 + 8 * ca + (8 / AR) * q, K - 8 / AR) * XSZ;
#pragma unroll
      for (int i = 0; i < AC; ++i) r.a[i][q] = load16_any(ap[i] + ka);
    }
    const int kb = min(k0 + 16 * cb, K - 16);
#pragma unroll
    for (int i = 0; i < BC; ++i) r.b[i] = load16_any(bp[i] + kb);
  };
  auto store = [&](Regs &r, int kt, int st) __attribute__((always_inline)) {
    uint8_t *const base = stages + st * G::STAGE;
    const int k0 = (kt0 + kt) * BK;
    if (k0 + BK > K) {  // the last tile: shift the clamped chunks into place
#pragma unroll
      for (int q = 0; q < AR; ++q) {
        const int k = k0 + 8 * ca + (8 / AR) * q, s = min(max(k - (K - 8 / AR), 0), 16) * XSZ;
#pragma unroll
        for (int i = 0; i < AC; ++i) r.a[i][q] = shr_bytes(r.a[i][q], s);
      }
      const int s = max(k0 + 16 * cb - (K - 16), 0);
#pragma unroll
      for (int i = 0; i < BC; ++i) r.b[i] = shr_bytes(r.b[i], s);
    }
#pragma unroll
    for (int i = 0; i < AC; ++i) {
      if constexpr (P == 3) {
        uint4 o[3];
        split8(r.a[i][0], r.a[i][1], o);
#pragma unroll
        for (int p = 0; p < 3; ++p) store16(base + p * G::A_PLANE + a_dst[i], o[p]);
      } else {
        store16(base + a_dst[i], r.a[i][0]);
      }
    }
#pragma unroll
    for (int i = 0; i < BC; ++i) store16(base + b_dst[i], r.b[i]);
  };

  f32x16 tot[BMB][BNB], hi[BMB][BNB], low[BMB][BNB];  // hi, low: fp32 activations only
#pragma unroll
  for (int i = 0; i < BMB; ++i)
#pragma unroll
    for (int j = 0; j < BNB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) tot[i][j][e] = hi[i][j][e] = low[i][j][e] = 0.f;

  const int a_row = (wm * 32 * BMB + l32) * 128, b_row = P * G::A_PLANE + (wn * 32 * BNB + l32) * 64;
  const int a_sw = (l32 >> 1) & 7, b_sw = (l32 >> 2) & 3;
  auto compute = [&](int st) __attribute__((always_inline)) {
    const uint8_t *const base = stages + st * G::STAGE;
    uint4 fb[BNB];
#pragma unroll
    for (int s = 0; s < 4; ++s) {  // 16 k each: sub-step 2p + h, lane group g: k chunk 4p + 2g + h
      const int c = 4 * (s >> 1) + 2 * g + (s & 1);
      uint4 fa[P][BMB], q[BNB];
      if ((s & 1) == 0)
#pragma unroll
        for (int j = 0; j < BNB; ++j)
          fb[j] = *reinterpret_cast<const uint4 *>(base + b_row + j * 2048 + (((2 * (s >> 1) + g) ^ b_sw) << 4));
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int i = 0; i < BMB; ++i)
          fa[p][i] = *reinterpret_cast<const uint4 *>(base + p * G::A_PLANE + a_row + i * 4096 + ((c ^ a_sw) << 4));
#pragma unroll
      for (int j = 0; j < BNB; ++j) q[j] = (s & 1) ? Ac::dq8(fb[j].z, fb[j].w) : Ac::dq8(fb[j].x, fb[j].y);
#pragma unroll
      for (int i = 0; i < BMB; ++i)
#pragma unroll
        for (int j = 0; j < BNB; ++j) {
          if constexpr (P == 3) {
            low[i][j] = Ac::mfma32(fa[2][i], q[j], low[i][j]);
            low[i][j] = Ac::mfma32(fa[1][i], q[j], low[i][j]);
            hi[i][j] = Ac::mfma32(fa[0][i], q[j], hi[i][j]);
          } else {
            tot[i][j] = Ac::mfma32(fa[0][i], q[j], tot[i][j]);
          }
        }
    }
  };
  auto fold = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < BMB; ++i)
#pragma unroll
      for (int j = 0; j < BNB; ++j) {
        tot[i][j] += hi[i][j];
#pragma unroll
        for (int e = 0; e < 16; ++e) hi[i][j][e] = 0.f;
      }
  };
  auto barrier = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  // ---- K loop: compute tile kt from LDS stage kt % 2 while tile kt + 1 waits
  // in registers (or arrives) and tile kt + 2 is requested. Loads past the
  // group's tiles are clamped like any other and never stored.
  // (No branch between the requests and the waits for them: where two paths
  // meet, the compiler waits for the stricter count, here for every load.)
  Regs r0, r1;
  load(r0, 0);
  load(r1, 1);
  store(r0, 0, 0);
  barrier();
  int kt = 0;
  for (; kt + kFold < n; kt += kFold) {
    load(r0, kt + 2);
    compute(0);
    store(r1, kt + 1, 1);
    barrier();
    load(r1, kt + 3);
    compute(1);
    if constexpr (P == 3) fold();
    store(r0, kt + 2, 0);
    barrier();
  }
  compute(0);
  if (kt + 1 < n) {
    store(r1, kt + 1, 1);
    barrier();
    compute(1);
  }
  if constexpr (P == 3) fold();
  if constexpr (P == 3)
#pragma unroll
    for (int i = 0; i < BMB; ++i)
#pragma unroll
      for (int j = 0; j < BNB; ++j) tot[i][j] += low[i][j];

  if constexpr (KG > 1) {
    // groups 1.. hand their sums to group 0 through LDS: [group][wave][block][quad][lane] of 16 bytes
    constexpr int BLK = BMB * BNB * 4;
    barrier();  // every wave is done with the stages
    f32x4 *const part = reinterpret_cast<f32x4 *>(lds);
    auto at = [&](int grp, int c) { return (((grp - 1) * WM * WN + wg) * BLK + c) * 64 + lane; };
    if (kg > 0) {
#pragma unroll
      for (int c = 0; c < BLK; ++c) {
        const f32x16 &a = tot[c / 4 / BNB][c / 4 % BNB];
        const int q = 4 * (c % 4);
        part[at(kg, c)] = f32x4{a[q], a[q + 1], a[q + 2], a[q + 3]};
      }
    }
    barrier();
    if (kg > 0) return;
#pragma unroll
    for (int grp = 1; grp < KG; ++grp)
#pragma unroll
      for (int c = 0; c < BLK; ++c) {
        const f32x4 v = part[at(grp, c)];
#pragma unroll
        for (int e = 0; e < 4; ++e) tot[c / 4 / BNB][c / 4 % BNB][4 * (c % 4) + e] += v[e];
      }
  }

  // ---- epilogue: lane (l32, g) holds column l32, rows (e & 3) + 8 * (e >> 2) + 4g
#pragma unroll
  for (int j = 0; j < BNB; ++j) {
    const int nn = n0 + (wn * BNB + j) * 32 + l32;
    if (nn >= N) continue;
    const float sn = scale[nn];
    const float bn = bias ? load_as_f32(bias, nn, bias_dt) : 0.f;
#pragma unroll
    for (int i = 0; i < BMB; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + (wm * BMB + i) * 32 + (e & 3) + 8 * (e >> 2) + 4 * g;
        float v = tot[i][j][e] * sn;
        if (bias) v += bn;
        if (m < M) store_from_f32(y, (int64_t)m * ldy + nn, XDT, v);
      }
  }
}

template <int XDT, int BMB, int BNB, int WM, int WN, int KG>
static void go(const GemmArgs &a, hipStream_t s) {
  using G = Geo<XDT, BMB, BNB, WM, WN, KG>;
  const int tm = (int)((a.M + G::BM - 1) / G::BM), tn = (int)((a.N + G::BN - 1) / G::BN);
  hipLaunchKernelGGL((staged_kernel<XDT, BMB, BNB, WM, WN, KG>), dim3((unsigned)(tm * tn)), dim3(G::THREADS), 0, s,
                     a.x, a.ldx, a.w, a.ldw, a.scale, a.bias, a.bias_dt, a.y, a.ldy, (int)a.M, (int)a.N, (int)a.K, tm,
                     tn);
}

}  // namespace staged

#ifdef RA_TUNING
extern int g_staged_cfg;  // tuning builds: forced geometry (index below)
#endif

bool staged_supported(const GemmArgs &a) {
  if (a.M < 1 || a.N < 1 || a.K < 16) return false;
  if (a.M > ((int64_t)1 << 30) || a.N > ((int64_t)1 << 30) || a.K > ((int64_t)1 << 29)) return false;
  return ((a.M + 31) / 32) * ((a.N + 31) / 32) < ((int64_t)1 << 22);  // one launch: at most 2^32 threads
}

// Where it is ahead of the VALU kernel (graph replay of cold weights, us, VALU
// kernel -> this): everywhere from 5 rows (fp32 M=8 K=N=1000 12.8 -> 8.9,
// M=16 K=N=4096 133.6 -> 24.3, fp16 M=8 K=1001 N=1000 12.7 -> 6.2), with
// fewer rows in 16 bits unless the weight is tiny (M=1 K=N=1000 6.5 -> 5.0,
// K=4100 N=8200 52.9 -> 18.6), in fp32, whose tiles convert 32 rows however
// few there are, from 2^23 weights at M = 1 and 2^22 at M = 2..4 (M=1
// K=N=4096 33.4 -> 23.2, M=2 K=2048 N=4096 16.1 -> 13.1; M=1 K=N=1000 7.0
// against 8.2).
bool staged_selected(const GemmArgs &a) {
  if (!staged_supported(a)) return false;
  if (a.M > 4) return true;
  const int64_t weights = a.N * a.K;
  if (a.x_dt != RA_F32) return weights >= ((int64_t)1 << 18);
  return weights >= ((int64_t)1 << (a.M == 1 ? 23 : 22));
}

// Geometry. fp32 (us, by the two below): 32 x 64 tiles in 4 K groups run one
// workgroup per CU and round at about 3.5 + 0.0052 K, 64 x 128 in 2 groups at
// 5 + 0.0145 K with four times the outputs (M=512 K=N=4096 96.9 / 69.0, M=128
// 26.9 / 56.1, M=512 K=300 N=4096 28.0 / 12.9, M=256 K=N=2048 16.2 / 30.7).
// 16 bits (no conversion, less LDS): the smallest tile that stays within
// about one round: 32 x 32 (M=2 K=2047 N=4096 9.0 against 10.7 with 32 x 64),
// 32 x 64 (M=77 K=1000 N=4101 8.3, 9.3 with 64 x 64), 64 x 64 (M=128 K=4100
// N=8200 38.4, 41.3 with 32 x 64), then 128 x 128 (M=512 72.8, 90.4 with
// 64 x 64; M=256 51.7, 54.8).
static int geometry(const GemmArgs &a) {
  auto tiles = [&](int bm, int bn) { return ((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn); };
  constexpr int64_t kCus = 256;
  if (a.x_dt == RA_F32) {
    const double small = (double)((tiles(32, 64) + kCus - 1) / kCus) * (3.5 + 0.0052 * (double)a.K);
    const double large = (double)((tiles(64, 128) + kCus - 1) / kCus) * (5.0 + 0.0145 * (double)a.K);
    return small <= large ? 1 : 2;
  }
  if (tiles(32, 32) <= kCus) return 3;
  if (tiles(32, 64) <= kCus + kCus / 4) return 4;
  return tiles(64, 64) <= kCus + kCus / 2 ? 5 : 6;
}

hipError_t staged_launch(const GemmArgs &a, hipStream_t s) {
  using namespace staged;
  int cfg = geometry(a);
#ifdef RA_TUNING
  if (g_staged_cfg) cfg = g_staged_cfg;
#endif
  if (a.x_dt == RA_F32) {
    if (cfg == 1) go<RA_F32, 1, 1, 1, 2, 4>(a, s);
    else go<RA_F32, 1, 2, 2, 2, 2>(a, s);
    return hipGetLastError();
  }
#define RA_STAGED(I_, ...)                                     \
  if (cfg == I_) {                                             \
    if (a.x_dt == RA_F16) go<RA_F16, __VA_ARGS__>(a, s);       \
    else go<RA_BF16, __VA_ARGS__>(a, s);                       \
    return hipGetLastError();                                  \
  }
  RA_STAGED(3, 1, 1, 1, 1, 4)  // 32 x 32, 4 groups
  RA_STAGED(4, 1, 1, 1, 2, 2)  // 32 x 64, 2 groups
  RA_STAGED(5, 1, 1, 2, 2, 1)  // 64 x 64
  RA_STAGED(6, 2, 2, 2, 2, 1)  // 128 x 128
#undef RA_STAGED
  return hipErrorInvalidValue;
}

}  // namespace ra
