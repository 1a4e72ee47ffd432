/*
 * Exhaustive check: orc_exp2f (the oracle's restatement of glibc's exp2f
 * algorithm) against the host libm exp2f on every float in [-151, 129],
 * which covers every input whose result is neither 0 nor +inf, and a sweep
 * of the special values outside it.  The same for the form of it that reduces
 * its argument in f32 (q3_device.h exp2f_fast), on every float in [-151, 200].
 * TEST INFRASTRUCTURE ONLY.
 * Prints "checked=N mismatches=M" and "fast checked=N mismatches=M" and exits
 * 0 iff both M == 0.
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#ifdef _OPENMP
#include <omp.h>
#endif

#include "ref_qwen3.h"

static float asf(uint32_t u) {
  float f;
  memcpy(&f, &u, 4);
  return f;
}
static uint32_t asu(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  return u;
}

static uint64_t tab[32]; /* bits(RN_double(2^(i/32))) - (i << 47) */

static float exp2f_fast(float x) {
  const float shift = 0x1.8p+18f;
  const float kf = x + shift;
  const uint32_t ki = asu(kf);
  const double r = (double)(x - (kf - shift));
  const uint64_t t = tab[ki & 31u] + ((uint64_t)(ki << 15) << 32);
  double s;
  memcpy(&s, &t, 8);
  const double z = fma(0x1.c6af84b912394p-5, r, 0x1.ebfce50fac4f3p-3);
  double y = fma(0x1.62e42ff0c52d6p-1, r, 1.0);
  y = fma(z, r * r, y);
  return (float)(y * s);
}

int main(void) {
  long long checked = 0, bad = 0, fchecked = 0, fbad = 0;
  for (int i = 0; i < 32; ++i) {
    const double v = (double)exp2l((long double)i / 32);
    memcpy(&tab[i], &v, 8);
    tab[i] -= (uint64_t)i << 47;
  }
#pragma omp parallel for reduction(+ : checked, bad, fchecked, fbad) schedule(static)
  for (long long hi = 0; hi < 65536; ++hi) {
    for (uint32_t lo = 0; lo < 65536; ++lo) {
      const uint32_t u = ((uint32_t)hi << 16) | lo;
      const float x = asf(u);
      if (x >= -151.0f && x <= 200.0f) {
        const float f = exp2f_fast(x);
        ++fchecked;
        if (asu(f) != asu(exp2f(x)) && ++fbad < 4) fprintf(stderr, "x=%a fast=%a libm=%a\n", x, f, exp2f(x));
      }
      const int inside = (x > -151.0f && x < 129.0f);
      /* outside the window only sample every 4096th pattern (+ specials) */
      if (!inside && (lo & 0xFFF) != 0 && !isnan(x) && !isinf(x)) continue;
      const float a = orc_exp2f(x), b = exp2f(x);
      ++checked;
      if (asu(a) != asu(b) && !(isnan(a) && isnan(b))) {
        ++bad;
        if (bad < 4) fprintf(stderr, "x=%a orc=%a libm=%a\n", x, a, b);
      }
    }
  }
  printf("checked=%lld mismatches=%lld\n", checked, bad);
  printf("fast checked=%lld mismatches=%lld\n", fchecked, fbad);
  return bad == 0 && fbad == 0 ? 0 : 1;
}
