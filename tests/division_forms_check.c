/*
 * The device's division (recip(), rdiv() in
 * fargo3d_amd/csrc/hip/f3d_device_body.h):
 *     r = estimate of 1/d, then twice r += r (1 - d r);
 *     q0 = RN(a r), rem = q0 d - a (one FMA), q = RN(q0 - rem r) (one FMA)
 * against IEEE division, in binary64 with the C library's fma.  The estimate
 * is 1/d with a relative error of up to 2^-BITS put on (the hardware's is
 * smaller).
 *
 *   division_forms_check N SEED BITS
 *     N random operand pairs, N pairs whose quotient lies next to a rounding
 *     midpoint, N exact quotients and N zeros of either sign, d > 0; prints
 *     "samples mismatches" (a mismatch is any differing bit)
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
static double unit(void) { return (double)(rnd() >> 11) * 0x1p-53; }
static double random_double(int positive) {
  double x = ldexp(1.0 + unit(), (int)(rnd() % 160) - 80);
  return positive || (rnd() & 1) ? x : -x;
}
static double bits_err;
static double device_div(double a, double d) {
  double r = (1.0 / d) * (1.0 + bits_err * (2.0 * unit() - 1.0));
  r = fma(fma(-d, r, 1.0), r, r);
  r = fma(fma(-d, r, 1.0), r, r);
  const double q0 = a * r;
  return fma(-fma(q0, d, -a), r, q0);
}
static long bad;
static void check(double a, double d) {
  const double q = device_div(a, d), w = a / d;
  if (memcmp(&q, &w, 8)) bad++;
}

int main(int argc, char **argv) {
  const long n = atol(argv[1]);
  s = (uint64_t)atoll(argv[2]) * 0x9E3779B97F4A7C15ull + 1;
  bits_err = ldexp(1.0, -atoi(argv[3]));
  if (argc < 4) return 2;
  for (long i = 0; i < n; i++) {
    double d = random_double(1);
    check(random_double(0), d);
    /* next to a midpoint: a = RN(d (q + half an ulp)) and its neighbours */
    const double q = random_double(0), h = 0.5 * (nextafter(q, INFINITY) - q);
    const double a = d * q + d * h;
    check(a, d);
    check(nextafter(a, INFINITY), d);
    check(nextafter(a, -INFINITY), d);
    /* exact quotients */
    const double d26 = ldexp((double)((rnd() & 0x3ffffff) | 1), (int)(rnd() % 40) - 20);
    const double q26 = ldexp((double)(int64_t)((rnd() & 0x3ffffff)) - 0x2000000, (int)(rnd() % 40) - 20);
    check(d26 * q26, d26);
    check(rnd() & 1 ? 0.0 : -0.0, d);
  }
  printf("%ld %ld\n", 6 * n, bad);
  return 0;
}
