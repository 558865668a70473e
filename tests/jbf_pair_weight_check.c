/* Intensity weight of the radius-4 joint bilateral filter in pairs of floats
 * (k_jbf_r4's arithmetic, operation for operation) against the reference
 * expressions: "div" compares the quotient with IEEE division, "exp" every
 * weight that the method keeps with (float)exp(-(double)di2 / kI) over the
 * floats di2 (every stride-th), and prints the largest error of the sum before
 * its last rounding as a fraction of the band that is not kept.
 *   cc -O2 -mfma -ffp-contract=off jbf_pair_weight_check.c -lm */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#define N 8192
static float thi[N], tlo[N];

static uint32_t bits(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static float fl(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }

static const float S = 0x1p22f - 0.25f, M = 0x1p22f - 0.5f;
static const float C1 = (float)(0x1.62e42fefa39efp-1 / N);
static const float C2 = (float)(0x1.62e42fefa39efp-1 / N * (0x1.62e42fefa39efp-1 / N) / 2);
static const float KEEP = 0x1p-24f - 0x1p-35f;

/* 1: kept, *h is the weight; 0: left to the reference expression */
static int weight(float di2, float nh, float nl, float far, float under, float *h, double *err) {
  const float sh = fmaf(di2, nh, S);
  *err = 0;
  const uint32_t b = bits(sh), n = b & 0xffff8000u;
  float f = fmaf(di2, nh, M - fl(b & ~3u));
  f = fmaf(di2, nl, f);
  const float q = f * fmaf(f, C2, C1);
  const int j = (b >> 2) & (N - 1);
  const float s = fmaf(thi[j], q, tlo[j]);
  const float v = thi[j] + s;
  const float e = s - (v - thi[j]);
  *h = fl(bits(v) + (n << 8));
  if (sh < under) {
    *h = 0.f;
    return 1;
  }
  const long double x = (long double)di2 * ((long double)nh + nl) - (fl(b & ~3u) - 0x1p22f - j);
  *err = (double)fabsl((long double)thi[j] + s + exp2l(x / N)) / 0x1p-35;
  if (sh >= far) return fabsf(e) <= KEEP;
  /* below 2^-125: round to a multiple of 2^-149 */
  const int k = (int)(n >> 15 & 0xff) - 256;
  *h = v * -0x1p-64f * fl((uint32_t)(127 + 64 + k) << 23);
  const float r = v + *h * 0x1p64f * fl((uint32_t)(127 - 64 - k) << 23);
  return fabsf(r + e) <= fl((uint32_t)(127 - 150 - k) << 23) * (1 - 0x1p-20f) - 0x1p-35f;
}

int main(int argc, char **argv) {
  long cases = 0, left = 0, bad = 0;
  double worst = 0;
  for (int j = 0; j < N; j++) {
    const long double t = exp2l((j + 0.5L) / N);
    thi[j] = (float)-t;
    tlo[j] = (float)(-t - thi[j]);
  }
  if (argc == 3 && !strcmp(argv[1], "div")) { /* significands of the divisor, several dividends each */
    uint64_t x = 88172645463325252ull;
    for (uint32_t i = 0; i < 1u << 23; i++) {
      const float m = fl(0x3f800000u | i), yh = 1.0f / m, yl = fmaf(-m, yh, 1.0f) * yh;
      for (int k = 0; k < atoi(argv[2]); k++) {
        x ^= x << 13, x ^= x >> 7, x ^= x << 17;
        const float a = fl(0x3f800000u | (uint32_t)(x >> 41));
        const float q = fmaf(a, yh, a * yl);
        bad += fmaf(fmaf(-q, m, a), yh, q) != a / m;
        cases++;
      }
    }
  } else { /* exp STRIDE SIGMA */
    const double kI = 2.0 * (double)(float)atof(argv[3]) * (2.0 * (double)(float)atof(argv[3]));
    const double n = -(double)N / 0x1.62e42fefa39efp-1 / kI;
    const float nh = (float)n, nl = (float)(n - nh);
    const float far = (float)(0x1p22 - 87.0 / 0x1.62e42fefa39efp-1 * N);
    const float under = (float)(0x1p22 - 104.5 / 0x1.62e42fefa39efp-1 * N);
    for (uint64_t u = 0; u <= bits((float)(110.0 * kI)); u += (uint64_t)atoi(argv[2])) {
      float h;
      double err;
      const float di2 = fl((uint32_t)u);
      const int kept = weight(di2, nh, nl, far, under, &h, &err);
      if (err > worst) worst = err;
      cases++;
      if (!kept) left++;
      else bad += bits(h) != bits((float)exp(-(double)di2 / kI));
    }
  }
  printf("%ld %ld %ld %.3f\n", cases, left, bad, worst);
  return 0;
}
