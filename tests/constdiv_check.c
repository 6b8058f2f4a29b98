/* CPU check of the FP32 division by the lattice constants y as two operations,
 *   q = fma(x, r, x * l),  r = RN(1/y), l = RN(1/y - r):
 * 1. q against the IEEE quotient x / y for every significand of x at biased
 *    exponents 51 (the smallest the kernels rely on), 52, 90, 127, 128, and
 *    for x = +0: between these the operations only scale with x;
 * 2. the equilibria (D2Q9, D2Q13) with this division against those with the
 *    IEEE division, for velocities with u.u < 1/2 of every size: zero,
 *    subnormal, tiny and ordinary components, ux = +-uy.
 * Prints, per constant and per lattice, what was tested and the mismatches. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static float bits(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static uint32_t ubits(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }

static float dv(int fast, float x, float y) {
  const float r = 1.0f / y, l = (float)(1.0 / (double)y - (double)r);
  return fast ? fmaf(x, r, x * l) : x / y;
}

static const int KX[13] = {0, 1, 0, -1, 0, 1, -1, -1, 1, 2, 0, -2, 0};
static const int KY[13] = {0, 0, 1, 0, -1, 1, 1, -1, -1, 0, 2, 0, -2};
static const int POS[6] = {1, 2, 5, 6, 9, 10}, NEG[6] = {3, 4, 7, 8, 11, 12};

/* brackets of the equilibrium (W rho is a common factor) */
static void eq(int q13, int fast, float ux, float uy, float *out) {
  const float C = 1.0f / sqrtf(q13 ? 2.0f : 3.0f);
  const float C2 = C * C, C4 = C2 * C2, C6 = C2 * C4;
  const float uu = ux * ux + uy * uy, D = dv(fast, uu, 2.0f * C2);
  out[0] = 1.0f - D;
  for (int i = 0; i < (q13 ? 6 : 4); ++i) {
    float cu = 0.0f; cu += (float)KX[POS[i]] * ux; cu += (float)KY[POS[i]] * uy;
    const float A = dv(fast, cu, C2), B = dv(fast, cu * cu, 2.0f * C4);
    float bp = ((1.0f + A) + B) - D, bn = ((1.0f - A) + B) - D;
    if (q13) {
      const float E = dv(fast, cu * (cu * cu), 2.0f * C6), G = dv(fast, (3.0f * cu) * uu, 2.0f * C4);
      bp = (bp + E) - G;
      bn = (bn - E) + G;
    }
    out[POS[i]] = bp;
    out[NEG[i]] = bn;
  }
}

static uint64_t seed = 88172645463325252ull;
static uint64_t rnd(void) { seed ^= seed << 13; seed ^= seed >> 7; return seed ^= seed << 17; }
static float component(void) {  /* 2^-149 .. 0.7, or zero */
  const uint64_t r = rnd();
  if (r % 16 == 0) return 0.0f;
  const float m = 1.0f + (float)(rnd() & 0x7fffff) / 8388608.0f;
  const int e = r % 3 == 0 ? -(int)(rnd() % 150) : -(int)(rnd() % 40);
  return ((r >> 8) & 1 ? -0.35f : 0.35f) * ldexpf(m, e);
}

int main(int argc, char **argv) {
  const long n = argc > 1 ? atol(argv[1]) : 1000000;
  const int exps[5] = {51, 52, 90, 127, 128};
  for (int q13 = 0; q13 < 2; ++q13) {
    const float C = 1.0f / sqrtf(q13 ? 2.0f : 3.0f);
    const float C2 = C * C, C4 = C2 * C2, C6 = C2 * C4, ys[4] = {C2, 2.0f * C4, 2.0f * C2, 2.0f * C6};
    for (int k = 0; k < (q13 ? 4 : 3); ++k) {
      long bad = ubits(dv(1, 0.0f, ys[k])) != 0;
      for (int e = 0; e < 5; ++e)
        for (uint32_t m = 0; m < (1u << 23); ++m) {
          const float x = bits(((uint32_t)exps[e] << 23) | m);
          bad += ubits(dv(1, x, ys[k])) != ubits(x / ys[k]);
        }
      printf("%.9g %ld %ld\n", ys[k], 5l << 23, bad);
    }
    long tested = 0, bad = 0;
    for (long i = 0; i < n; ++i) {
      float ux = component(), uy = component(), a[13], b[13];
      const int kind = (int)(rnd() % 8);
      if (kind < 2) uy = kind ? ux : -ux;
      if (!(ux * ux + uy * uy < 0.5f)) continue;
      eq(q13, 1, ux, uy, a);
      eq(q13, 0, ux, uy, b);
      ++tested;
      bad += memcmp(a, b, (q13 ? 13 : 9) * sizeof(float)) != 0;
    }
    printf("d2q%d %ld %ld\n", q13 ? 13 : 9, tested, bad);
  }
  return 0;
}
