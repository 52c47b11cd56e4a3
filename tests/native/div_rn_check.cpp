/* Exhaustive-by-sampling check of the kernels' divisions and square roots
 * (gmcore_amd/csrc/gmc_arith.hpp, the code itself):
 *   div_rn     from y = 1 / d correctly rounded must equal the IEEE quotient
 *              (a zero numerator gives a zero; -0 / d may be +0);
 *   div_from   the same from an estimate of 1 / d up to 2^-22 off;
 *   sqrt_from  the IEEE square root for 0 and x >= 1e-290 from an estimate of
 *              1 / sqrt(x) up to 2^-22 off.
 *
 * usage: div_rn_check DENOMS_FILE SAMPLES_PER_DENOM SEED
 * DENOMS_FILE holds raw doubles (the divisor metric terms of real meshes);
 * adversarial divisors (powers of two, all-ones and one-ulp-above-one
 * significands) are added here.  For each divisor the numerators are random
 * doubles over 200 binades and, for the hard cases of rounding, a = RN(d m)
 * and its four nearest neighbours for random rounding midpoints m (d m is
 * exact in binary128), so that a / d lies within a few ulps of 2^-53 of a
 * midpoint; square roots are taken of random doubles over 1800 binades and of
 * the doubles around the squares of doubles and of midpoints.  Prints
 * "checked N mismatches M" and exits 1 on a mismatch. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "../../gmcore_amd/csrc/gmc_arith.hpp"

using gmc::div_from;
using gmc::div_rn;
using gmc::sqrt_from;

static uint64_t st;
static uint64_t rnd(void) {
  st ^= st << 13;
  st ^= st >> 7;
  st ^= st << 17;
  return st;
}
static double from_bits(uint64_t b) {
  double x;
  memcpy(&x, &b, 8);
  return x;
}
static uint64_t bits(double x) {
  uint64_t b;
  memcpy(&b, &x, 8);
  return b;
}
static double rdbl(int e0, int span) {
  return from_bits((rnd() & 0x000fffffffffffffull) | ((uint64_t)(1023 + e0 + (int)(rnd() % (uint64_t)span)) << 52));
}
static long checked, bad;
static void expect(const char *what, double a, double d, double want, double got) {
  checked++;
  if (bits(want) != bits(got) && !(want == 0.0 && got == 0.0)) {
    if (bad < 5) printf("%s mismatch a=%a d=%a want=%a got=%a\n", what, a, d, want, got);
    bad++;
  }
}
/* an estimate of x as the hardware may give it */
static double rough(double x) {
  const double err = ldexp((double)(rnd() % 2001) / 1000.0 - 1.0, -22);
  return x * (1.0 + err);
}
static void check(double a, double d, double y) {
  const double want = a / d;
  expect("div_rn", a, d, want, div_rn(a, d, y));
  expect("div_from", a, d, want, div_from(a, d, rough(y)));
}
static void check_sqrt(double x) {
  expect("sqrt_from", x, 0.0, sqrt(x), sqrt_from(x, rough(1.0 / sqrt(fmax(x, 1e-290)))));
}

static void one_divisor(double d, long n) {
  const double y = 1.0 / d;
  check(0.0, d, y);
  check(-0.0, d, y);
  for (long k = 0; k < n; k++) {
    double a = rdbl(-100, 200);
    check((rnd() & 1) ? -a : a, d, y);
    /* near-midpoint quotients: a / d ~ q + ulp(q) / 2 */
    const double q = rdbl(-40, 80);
    const __float128 m = (__float128)q + ((__float128)nextafter(q, INFINITY) - (__float128)q) / 2;
    const double a0 = (double)((__float128)d * m);
    for (int off = -2; off <= 2; off++) check(from_bits(bits(a0) + (int64_t)off), d, y);
  }
}

int main(int argc, char **argv) {
  if (argc < 4) return 2;
  const long n = atol(argv[2]);
  st = 0x9E3779B97F4A7C15ull ^ (uint64_t)atol(argv[3]);
  FILE *f = fopen(argv[1], "rb");
  if (!f) return 2;
  double d;
  long nd = 0;
  while (fread(&d, sizeof d, 1, f) == 1) {
    if (d != 0.0 && isfinite(d)) { one_divisor(d, n); nd++; }
  }
  fclose(f);
  for (int e = -30; e <= 30; e += 3) {
    one_divisor(ldexp(1.0, e), n);
    one_divisor(ldexp(2.0 - ldexp(1.0, -52), e), n);
    one_divisor(ldexp(1.0 + ldexp(1.0, -52), e), n);
    one_divisor(-ldexp(1.5, e), n);
    nd += 4;
  }
  check_sqrt(0.0);
  for (long k = 0; k < 500 * n; k++) {
    check_sqrt(rdbl(-960, 1900));
    const double g = rdbl(-450, 900);
    const __float128 m = (__float128)g + ((__float128)nextafter(g, INFINITY) - (__float128)g) / 2;
    const double x0 = g * g, x1 = (double)(m * m);
    for (int off = -2; off <= 2; off++) {
      check_sqrt(from_bits(bits(x0) + (int64_t)off));
      check_sqrt(from_bits(bits(x1) + (int64_t)off));
    }
    const double tiny = rdbl(-1022, 57);   /* below 1e-290 */
    const double r = sqrt_from(tiny, rough(1.0 / sqrt(fmax(tiny, 1e-290))));
    checked++;
    if (tiny < 1e-290 && !(fabs(r) < 1e-140)) bad++;
  }
  printf("divisors %ld checked %ld mismatches %ld\n", nd, checked, bad);
  return bad != 0;
}
