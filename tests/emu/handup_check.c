/*
 * handup_check.c -- host replay of the register form's bound-set recurrence
 * (unbind_resident of ahf_amd/csrc/unbind_gpu.hip): wavefronts of 64 threads
 * of 8 members each, every thread in order, every wavefront until none of its
 * statuses changes, and the wavefronts' totals handed up until none below the
 * last has changed (ahf_handup_moved of unbind_core.h).  Velocities are
 * multiples of 1/16, so sums are exact in any order, with NaN, infinities and
 * very large values put into the first, a middle or the last wavefront, alone
 * and together.  The statuses must be the sequential loop's, after at most
 * one round more than there are wavefronts.
 *
 * usage: handup_check [runs] [seed]
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "../../ahf_amd/csrc/unbind_core.h"

#define IPT 8
#define MAX_NW 8

static uint64_t rs = 88172645463325252ull;
static uint64_t xr(void)
{
  rs ^= rs << 13;
  rs ^= rs >> 7;
  rs ^= rs << 17;
  return rs;
}
static double ur(void) { return (double)(xr() >> 11) * (1.0 / 9007199254740992.0); }

typedef struct {
  double x, y, m;
} tot;

static int n, nw;
static double vx[MAX_NW * 64 * IPT], vy[MAX_NW * 64 * IPT], lim[MAX_NW * 64 * IPT];
static uint32_t alive[MAX_NW * 64];

static int bound(int j, tot V)
{
  const double dx = vx[j] - V.x / V.m, dy = vy[j] - V.y / V.m;
  return !(dx * dx + dy * dy > lim[j]);
}

static tot wave_total(int w, const uint32_t *b)
{
  tot s = {0, 0, 0};
  for (int l = 0; l < 64; l++)
    for (int i = 0; i < IPT; i++)
      if ((b[64 * w + l] >> i) & 1u) {
        const int j = (64 * w + l) * IPT + i;
        s.x += vx[j];
        s.y += vy[j];
        s.m += 1.0;
      }
  return s;
}

/* one wavefront until none of its statuses changes; returns the evaluations */
static int wave_settle(int w, tot base, uint32_t *b)
{
  for (int sweeps = 1;; sweeps++) {
    uint32_t nb[64];
    int changed = 0;
    tot ex = base;
    for (int l = 0; l < 64; l++) {
      tot V = ex; /* the lower lanes' last statuses */
      nb[l] = 0;
      for (int i = 0; i < IPT; i++) {
        const int t = 64 * w + l, j = t * IPT + i;
        if (!((alive[t] >> i) & 1u)) continue;
        if (bound(j, V)) {
          nb[l] |= 1u << i;
          V.x += vx[j];
          V.y += vy[j];
          V.m += 1.0;
        }
      }
      for (int i = 0; i < IPT; i++)
        if ((b[64 * w + l] >> i) & 1u) {
          const int j = (64 * w + l) * IPT + i;
          ex.x += vx[j];
          ex.y += vy[j];
          ex.m += 1.0;
        }
    }
    for (int l = 0; l < 64; l++) {
      changed |= nb[l] != b[64 * w + l];
      b[64 * w + l] = nb[l];
    }
    if (!changed || sweeps > 66) return sweeps;
  }
}

int main(int argc, char **argv)
{
  const long runs = argc > 1 ? atol(argv[1]) : 2000;
  if (argc > 2) rs ^= (uint64_t)atoll(argv[2]) * 0x9E3779B97F4A7C15ull;
  const double odd[4] = {NAN, INFINITY, -INFINITY, 1e30};
  long bad = 0, many = 0;
  for (long run = 0; run < runs; run++) {
    nw = (run & 1) ? 8 : 4;
    n = nw * 64 * IPT - (int)(xr() % (64 * IPT));
    if (run % 5 == 0) n = (nw - 1) * 64 * IPT + 1;
    memset(alive, 0, sizeof(alive));
    const double scale = (double)(1 + xr() % 64) / 16.0;
    for (int j = 0; j < n; j++) {
      alive[j / IPT] |= 1u << (j % IPT);
      vx[j] = floor(64.0 * scale * (ur() + ur() - 1.0)) / 16.0;
      vy[j] = floor(64.0 * scale * (ur() + ur() - 1.0)) / 16.0 + 3.0;
      lim[j] = (xr() % 40) ? 16.0 * scale * scale * (0.2 + ur()) : INFINITY;
    }
    for (int k = (int)(run % 4); k > 0; k--) {
      const int w = xr() % 3 == 0 ? 0 : (xr() & 1) ? nw - 1 : 1 + (int)(xr() % (unsigned)(nw - 2));
      const int lo = w * 64 * IPT, hi = (w + 1) * 64 * IPT < n ? (w + 1) * 64 * IPT : n;
      const int j = lo + (int)(xr() % (unsigned)(hi - lo));
      (xr() & 1 ? vx : vy)[j] = odd[xr() % 4];
      if (xr() & 1) lim[j] = INFINITY;
    }
    const tot seed = {vx[0], vy[0], 1.0};
    /* the sequential loop */
    uint32_t ref[MAX_NW * 64];
    memset(ref, 0, sizeof(ref));
    tot V = seed;
    for (int j = 0; j < n; j++)
      if (bound(j, V)) {
        ref[j / IPT] |= 1u << (j % IPT);
        V.x += vx[j];
        V.y += vy[j];
        V.m += 1.0;
      }
    /* the hand-up */
    uint32_t b[MAX_NW * 64];
    tot T[2][MAX_NW];
    memcpy(b, alive, sizeof(b));
    for (int w = 0; w < nw; w++) T[0][w] = wave_total(w, b);
    int round = 1, any = 1, sweeps = 0;
    for (;; round++) {
      any = 0;
      for (int w = 0; w < nw; w++) {
        tot base = seed;
        for (int k = 0; k < w; k++) {
          base.x += T[(round - 1) & 1][k].x;
          base.y += T[(round - 1) & 1][k].y;
          base.m += T[(round - 1) & 1][k].m;
        }
        uint32_t was[64];
        memcpy(was, b + 64 * w, sizeof(was));
        const int s = wave_settle(w, base, b);
        sweeps = s > sweeps ? s : sweeps;
        T[round & 1][w] = wave_total(w, b);
        for (int l = 0; l < 64; l++)
          if (w + 1 < nw) any |= ahf_handup_moved(was[l], b[64 * w + l]);
      }
      if (!any || round > nw + 1) break;
    }
    many += round > 2;
    if (any || sweeps > 65 || memcmp(b, ref, sizeof(b))) {
      if (bad < 10) fprintf(stderr, "run %ld: %d members, %d rounds, %d evaluations, %s\n", run, n, round, sweeps, any ? "no end" : "statuses differ");
      bad++;
    }
  }
  printf("{\"runs\": %ld, \"several_rounds\": %ld, \"bad\": %ld}\n", runs, many, bad);
  return bad != 0 || many * 4 < runs;
}
