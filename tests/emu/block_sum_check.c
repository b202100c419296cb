/*
 * block_sum_check.c -- host check of the heavy deposit's block sum
 * (ahf_amd/csrc/amr_core.h, ahf_fold_step and ahf_fold_block_in) against
 * AHF's sequential accumulation d = (float)((double)d + c): wherever every
 * contribution of a block has a step, none is negative and the sum of the
 * steps stays in the binade, the value must be the sequential one, bit for
 * bit, for blocks of 1 to 4096 contributions, from starts on, beside and
 * between binade edges of both signs, with steps of exact halves and of
 * halves off by one unit of the double sum, and blocks that end on the edge.
 * The same contributions 64 at a time through the fold of a block that the
 * test refuses (heavy_fold1 of amr_gpu.hip), except its hand-over at ties.
 * Exit status 0 when no accepted block differs and most plain ones are taken.
 *
 * usage: block_sum_check [runs] [seed]
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "../../ahf_amd/csrc/amr_core.h"

static uint64_t rs = 88172645463325252ull;
static uint64_t xr(void)
{
  rs ^= rs << 13;
  rs ^= rs >> 7;
  rs ^= rs << 17;
  return rs;
}
static double ur(void) { return (double)(xr() >> 11) * (1.0 / 9007199254740992.0); }

/* heavy_fold1 of amr_gpu.hip replayed lane by lane over [0, mm); *tie is set
 * where it would go on with fold_wave (an exact tie or a NaN), which
 * fold_check.c replays */
static float fold1(float d, const double *cv, int mm, int *tie)
{
  *tie = 0;
  for (int start = 0; start < mm;) {
    int normal, bad = start;
    const int e = ahf_fold_exponent(d, &normal);
    if (normal) {
      const double scale = ldexp(1.0, 23 - e);
      const int32_t K0 = (int32_t)ahf_fold_K(d, e);
      int32_t P = 0, before = 0;
      int ok = 1;
      for (bad = start; bad < mm; bad++) {
        int32_t r;
        ok = ahf_fold_step(cv[bad], scale, &r);
        before = P;
        P += r;
        const int32_t K = K0 + P, A = K < 0 ? -K : K;
        if (!(ok && A > (1 << 23) && A < (1 << 24) && (K ^ K0) >= 0)) break;
        before = P;
      }
      if (bad > start) d = (float)ldexp((double)(K0 + before), e - 23);
      if (bad == mm) break;
      if (!ok && !(fabs(cv[bad] * scale) >= 4194304.0)) {
        *tie = 1;
        return d;
      }
    }
    d = (float)((double)d + cv[bad]);
    start = bad + 1;
  }
  return d;
}

int main(int argc, char **argv)
{
  const long runs = argc > 1 ? atol(argv[1]) : 100000;
  if (argc > 2) rs ^= (uint64_t)atoll(argv[2]) * 0x9E3779B97F4A7C15ull;
  static double c[4096];
  long taken = 0, plain = 0, plain_taken = 0, bad = 0;
  for (long t = 0; t < runs; t++) {
    const int m = 1 + (int)(xr() % ((xr() & 7) ? 64 : 4096));
    /* K in [2^23, 2^24) times 2^(e-23), either sign */
    const int e = (xr() & 15) ? (int)(xr() % 60) - 20 : (int)(xr() % 254) - 126;
    int64_t K;
    switch (xr() % 4) {
    case 0: K = ((int64_t)1 << 23) + (int64_t)(xr() % 4); break;
    case 1: K = ((int64_t)1 << 24) - 1 - (int64_t)(xr() % 2000); break;
    default: K = ((int64_t)1 << 23) + (int64_t)(xr() % (1u << 23)); break;
    }
    if (xr() & 1) K = -K;
    const float d0 = (float)ldexp((double)K, e - 23);
    const int kind = (int)(xr() % 6);
    for (int i = 0; i < m; i++) {
      double x; /* in units of the value's ulp */
      switch (kind) {
      case 0: x = ur() * 4000.0; break;
      case 1: x = ur(); break;
      case 2: x = (double)(xr() % 64) / 2.0; break;                            /* halves: ties */
      case 3: x = (double)(xr() % 64) / 2.0 + ldexp((double)(xr() % 5) - 2.0, -30); break;
      case 4: x = (xr() & 1) ? 0.0 : ldexp(ur(), (int)(xr() % 60) - 36); break;
      default: x = (xr() % 50) ? ur() : -ur(); break;
      }
      c[i] = ldexp(x, e - 23);
    }
    {
      const int mm = m < 64 ? m : 64;
      const float st = (xr() & 7) ? d0 : (xr() & 1 ? -1.0f : 0.0f);
      int tie;
      const float f = fold1(st, c, mm, &tie);
      float a = st;
      for (int i = 0; i < mm; i++) a = (float)((double)a + c[i]);
      if (!tie && memcmp(&a, &f, 4)) {
        if (bad < 10) fprintf(stderr, "run %ld kind %d mm %d start %.9g: %.9g, fold %.9g\n", t, kind, mm, (double)st, (double)a, (double)f);
        bad++;
      }
    }
    if (kind == 0) plain += m < 1000 && K > 0 && K < (3 << 22);
    int ok = 1, normal;
    int64_t S = 0;
    const int ed = ahf_fold_exponent(d0, &normal);
    if (!normal || ed != e) continue; /* e = -127 */
    const double scale = ldexp(1.0, 23 - e);
    for (int i = 0; i < m && ok; i++) {
      int32_t r;
      ok = ahf_fold_step(c[i], scale, &r) && c[i] >= 0.0;
      S += r;
    }
    if (!ok || !ahf_fold_block_in(K, S)) continue;
    taken++;
    if (kind == 0) plain_taken += m < 1000 && K > 0 && K < (3 << 22);
    float a = d0;
    for (int i = 0; i < m; i++) a = (float)((double)a + c[i]);
    const float b = (float)ldexp((double)(K + S), e - 23);
    if (memcmp(&a, &b, 4)) {
      if (bad < 10) fprintf(stderr, "run %ld kind %d m %d K %lld e %d: %.9g, block %.9g\n", t, kind, m, (long long)K, e, (double)a, (double)b);
      bad++;
    }
  }
  printf("{\"runs\": %ld, \"taken\": %ld, \"plain\": %ld, \"plain_taken\": %ld, \"mismatches\": %ld}\n", runs, taken,
         plain, plain_taken, bad);
  return bad || plain_taken * 10 < plain * 9;
}
