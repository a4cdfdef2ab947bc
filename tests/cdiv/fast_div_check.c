/* Checks the FP64 reciprocal, quotient and root steps of the device code
 * (recip_fast, recip_rn, quot_r, sqrt_fast in flash5_amd/csrc/fx_device.hpp)
 * against IEEE division and square root.  The device starts from its hardware
 * reciprocal and root estimates, good to about 2^-24; here the starts are the
 * rounded values off by any relative error up to 2^-23.  For a divisor whose
 * significand is all ones the start has to lie above the reciprocal, which is a
 * hair above the midpoint of two doubles, and gfx950's does: on the device
 * every divisor of that significand (exponents -60..60, the 15 neighbours
 * below included) gives the IEEE bits, as it does with the compiler's division.
 * Prints "<name> <samples> <mismatches>" per step. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static uint64_t s = 0x9E3779B97F4A7C15ull;
static uint64_t next(void) {  /* splitmix64 */
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
static double from_bits(uint64_t b) { double d; memcpy(&d, &b, 8); return d; }

/* significands random, at both ends of the binade, or short; exponents within
 * span of zero */
static double sample(int span) {
  uint64_t m = next(), sig = m & 0xFFFFFFFFFFFFFull;
  const int kind = (int)(m >> 52) & 7;
  if (kind == 0) sig = 0xFFFFFFFFFFFFFull - (sig & 15);
  if (kind == 1) sig &= 15;
  if (kind == 2) sig &= 0xFFFFFFFF00000ull;
  const int e = (int)(next() % (uint64_t)(2 * span + 1)) - span;
  return from_bits(((uint64_t)(1023 + e) << 52) | sig);
}
static double off(double x) {  /* x (1 + d), |d| <= 2^-23 */
  return x * (1.0 + ((double)(int64_t)next() * 0x1p-63) * 0x1p-23);
}

static double recip_fast(double y) {
  double r0 = off(1.0 / y);
  uint64_t b;
  memcpy(&b, &y, 8);
  if ((b & 0xFFFFFFFFFFFFFull) == 0xFFFFFFFFFFFFFull)
    r0 = 1.0 / y * (1.0 + fabs(off(0x1p-25)));
  const double e = fma(-y, r0, 1.0);
  return fma(r0, fma(e, e, e), r0);
}
static double recip_rn(double y) {
  const double r = recip_fast(y);
  return fma(fma(-y, r, 1.0), r, r);
}
static double quot_r(double x, double y, double r) {
  const double q = x * r;
  return fma(fma(-y, q, x), r, q);
}
static double sqrt_fast(double x) {
  const double r = off(1.0 / sqrt(x));
  double g = x * r, h = 0.5 * r;
  const double d = fma(-h, g, 0.5);
  g = fma(g, d, g);
  h = fma(h, d, h);
  g = fma(fma(-g, g, x), h, g);
  return fma(fma(-g, g, x), h, g);
}

int main(int argc, char** argv) {
  const long n = argc > 1 ? atol(argv[1]) : 10000000;
  long bad[4] = {0, 0, 0, 0};
  const char* name[4] = {"recip_rn", "quot", "quot_shared", "sqrt"};
  for (long i = 0; i < n; ++i) {
    const double x = (i & 1) ? sample(400) : -sample(400), y = sample(400);
    const double r = recip_rn(y), f = recip_fast(y);
    bad[0] += r != 1.0 / y;
    bad[1] += quot_r(x, y, f) != x / y;
    bad[2] += quot_r(x, y, r) != x / y;
    bad[3] += sqrt_fast(y) != sqrt(y);
  }
  long total = 0;
  for (int k = 0; k < 4; ++k) {
    printf("%s %ld %ld\n", name[k], n, bad[k]);
    total += bad[k];
  }
  return total != 0;
}
