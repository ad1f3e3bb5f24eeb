/*
 * Sampled check of the division-free fp32 quotient of the per-channel weight
 * quantiser (rotalabs-accel_amd/csrc/ra_rowops.hip):
 *
 *   r = RN(1 / s), q0 = RN(x * r), q1 = fma(fma(-q0, s, x), r, q0),
 *   q2 = fma(fma(-q1, s, x), r, q1)
 *
 * q2 must equal RN(x / s) for every scale s >= 2^-90 of a finite row and every
 * |x| <= 127.5 * s: random pairs, and for random s the x nearest to the ties
 * (k + 1/2) * s, where a wrong last bit would move the rounded integer. Where
 * |x / s| < 1/4 only the rounded integer (0) matters and is compared.
 *
 * Built by tests/test_gpu_rowops.py with -ffp-contract=off; prints the
 * mismatch count and exits non-zero on any mismatch.
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>

static uint64_t state = 88172645463325252ull;
static uint32_t rnd(void) {
  state ^= state << 13;
  state ^= state >> 7;
  state ^= state << 17;
  return (uint32_t)(state >> 32);
}
static int wrong(float x, float s) {
  const float r = 1.0f / s, q0 = x * r;
  const float q1 = fmaf(fmaf(-q0, s, x), r, q0);
  const float q2 = fmaf(fmaf(-q1, s, x), r, q1);
  const float q = x / s;
  return fabsf(q) < 0.25f ? rintf(q2) != rintf(q) : q2 != q;
}

int main(void) {
  long bad = 0, n = 0;
  for (int i = 0; i < 2000000; ++i) {
    const int e = i % 5 == 0 ? (int)(rnd() % 210) - 90 : (int)(rnd() % 30) - 20;
    const float s = ldexpf(1.0f + (float)(rnd() >> 9) * 0x1p-23f, e);
    const float t = ((float)(rnd() % 127) + 0.5f) * s;
    float x = nextafterf(nextafterf(t, 0), 0);
    for (int k = 0; k < 5; ++k, ++n) {
      bad += wrong(x, s) + wrong(-x, s);
      x = nextafterf(x, INFINITY);
    }
    for (int k = 0; k < 4; ++k, ++n) bad += wrong(ldexpf((float)(rnd() >> 8), -24) * 127.5f * s, s);
    bad += wrong(ldexpf((float)(rnd() >> 8), -24 - (int)(rnd() % 60)) * s, s);
  }
  printf("%ld mismatches of %ld\n", bad, n);
  return bad != 0;
}
