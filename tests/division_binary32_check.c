/*
 * The device's division (recip(), rdiv() in
 * fargo3d_amd/csrc/hip/f3d_device_body.h) in binary32:
 *     r = estimate of 1/d, then twice r += r (1 - d r);
 *     q0 = RN(a r), rem = q0 d - a (one FMA), q = RN(q0 - rem r) (one FMA)
 * with the C library's fmaf and an estimate one unit in the last place below,
 * at or above RN(1/d) (the hardware's is within one unit).
 *
 *   division_binary32_check MODE STEP SEED
 *     range    every STEP-th significand of d in [1, 2), the exponents of d and
 *              a drawn with d and 1/d normal and |a| >= 2^-102: a random a, the
 *              three next to a rounding midpoint of the quotient, an exact
 *              quotient, a zero of either sign; counts differing bits from a / d
 *     small    the same with |a| below 2^-102; counts quotients more than one
 *              unit from a / d
 *     outside  a or d infinite or NaN, d = 0, d subnormal, a quotient that
 *              overflows; counts quotients that are not NaN
 *   prints "samples faults"
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static uint64_t s;
static uint64_t rnd(void) {
  s ^= s << 13;
  s ^= s >> 7;
  s ^= s << 17;
  return s;
}
static float mantissa(uint32_t m) { return 1.0f + (float)(m & 0x7fffff) * 0x1p-23f; }
static float moved(float x, int ulps) {
  for (; ulps > 0; ulps--) x = nextafterf(x, INFINITY);
  for (; ulps < 0; ulps++) x = nextafterf(x, -INFINITY);
  return x;
}
static float estimate(float d, int ulps) {
  /* a subnormal divisor is taken for zero, as the hardware's reciprocal does */
  if (fabsf(d) < 0x1p-126f) return copysignf(INFINITY, d);
  const float r = 1.0f / d;
  return isfinite(r) && r != 0.0f ? moved(r, ulps) : r;
}
static float device_div(float a, float d, int ulps) {
  float r = estimate(d, ulps);
  r = fmaf(fmaf(-d, r, 1.0f), r, r);
  r = fmaf(fmaf(-d, r, 1.0f), r, r);
  const float q0 = a * r;
  return fmaf(-fmaf(q0, d, -a), r, q0);
}
static long samples, bad;
static int mode;
static void check(float a, float d, int ulps) {
  const float q = device_div(a, d, ulps), w = a / d;
  samples++;
  if (mode == 0) bad += memcmp(&q, &w, 4) != 0;
  else if (mode == 1) bad += !(q >= nextafterf(w, -INFINITY) && q <= nextafterf(w, INFINITY));
  else bad += q == q;
}

int main(int argc, char **argv) {
  if (argc < 4) return 2;
  mode = argv[1][0] == 'r' ? 0 : argv[1][0] == 's' ? 1 : 2;
  const uint32_t step = (uint32_t)atol(argv[2]);
  s = (uint64_t)atoll(argv[3]) * 0x9E3779B97F4A7C15ull + 1;
  for (uint32_t m = 0; m < 1u << 23; m += step) {
    const int ulps = (int)(rnd() % 3) - 1;
    const float d1 = mantissa(m);
    if (mode == 2) {
      const float d = ldexpf(d1, (int)(rnd() % 240) - 120), a = rnd() & 1 ? d : -d;
      const float tiny = ldexpf((float)(rnd() % 0x7fffff + 1), -149);
      check(copysignf(INFINITY, a), d, ulps);
      check(NAN, d, ulps);
      check(a, 0.0f, ulps);
      check(0.0f, 0.0f, ulps);
      check(a, INFINITY, ulps);
      check(a, NAN, ulps);
      check(a, tiny, ulps);
      check(ldexpf(d1, 100), ldexpf(d1, -60), ulps);
      continue;
    }
    /* exponents: d and 1/d normal; the quotient normal */
    const int ed = (int)(rnd() % 200) - 100;
    const int lo = mode ? -126 : -102, hi = mode ? -103 : 120;
    int ea = lo + (int)(rnd() % (hi - lo + 1));
    if (ea - ed > 120) ea = ed + 120;
    if (ea - ed < -120) continue;
    const float d = ldexpf(d1, ed), q = mantissa((uint32_t)rnd());
    const float a = ldexpf(mantissa((uint32_t)rnd()), ea);
    check(rnd() & 1 ? a : -a, d, ulps);
    /* the binary32 numbers around d1 (q + half a unit of q) */
    const float mid = (float)((double)d1 * ((double)q + 0x1p-24));
    for (int k = -1; k <= 1; k++) check(ldexpf(moved(mid, k), ea), d, ulps);
    /* an exact quotient */
    const float d12 = (float)((rnd() & 0xfff) | 0x801), q11 = (float)((rnd() & 0x7ff) | 0x401);
    if (!mode) check(ldexpf(d12 * q11, ea - 21), ldexpf(d12, ed - 11), ulps);
    check(rnd() & 1 ? 0.0f : -0.0f, d, ulps);
  }
  printf("%ld %ld\n", samples, bad);
  return 0;
}
