/*
 * amr_gpu.hip -- device pipeline of AHF's AMR hierarchy on gfx950.
 *
 * One call builds what src/main.c:614-648 builds on the CPU (gen_domgrids,
 * ll, zero_dens + assign_npart, the recursive gen_AMRhierarchy with
 * refine_grid / relink / relink_back), level by level, with everything
 * resident in HBM.  Per level the kernels are:
 *
 *   k_pmask        presence mask of every node (get_TSCnodes rules)
 *   k_prep         TSC weights and position of every bucket entry (k_prep_q:
 *                  the position alone, on levels that march or walk per source)
 *   k_gather_full  exact-order TSC density (assign_npart) of a level that holds
 *                  every octet, marching through its planes
 *   k_gather_light the same on the others, one lane per node (k_gather_src:
 *                  many entries per node)
 *   k_gather_heavy the same, nodes with many contributions, by wavefronts
 *   k_flags        interior + refinement criterion (test_node)
 *   k_refine_rows  ref_pquad/ref_cquad/ref_nquad block tests and run state
 *                  machine, one thread per level row
 *   scans +
 *   k_compact      octets of the next level, sorted (z,y,x)
 *   k_nbr_next     27-octet neighbour table of the next level
 *   k_relink_child particles to the first interior child containing them
 *   k_fine_count,  the fine buckets, each filled from its mother's bucket
 *   k_fine_fill    in bucket order
 *
 * The per-thread rules live in amr_core.h.  The domain level is binned by a
 * stable LSD radix sort (devprims.h) so every node's bucket is in particle
 * order, which fixes AHF's list order and hence its FP32 summation order.
 */
#include <hip/hip_runtime.h>

#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "../../include/ahf_gpu.h"
#include "amr_core.h"
#include "devprims.h"
#include "gpu_ctx.h"
#include "level_host.h"

using namespace ahf;

/* ================================================================ kernels */

__global__ void k_domain_octets(int64_t half, uint64_t *__restrict__ key, uint8_t *__restrict__ link,
                                int32_t *__restrict__ nbr)
{
  const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t no = half * half * half;
  if (o >= no) return;
  const int64_t ox = o % half, oy = (o / half) % half, oz = o / (half * half);
  key[o] = ahf_pack3((uint64_t)ox, (uint64_t)oy, (uint64_t)oz);
  link[o] = ox < half - 1 ? 1 : 0;
  for (int ez = -1; ez <= 1; ez++)
    for (int ey = -1; ey <= 1; ey++)
      for (int ex = -1; ex <= 1; ex++) {
        const int64_t nx = ahf_wrap(ox + ex, half), ny = ahf_wrap(oy + ey, half), nz = ahf_wrap(oz + ez, half);
        nbr[27 * o + ahf_e27(ex, ey, ez)] = (int32_t)((nz * half + ny) * half + nx);
      }
}

__global__ void k_domain_rows(int64_t half, uint64_t *__restrict__ row_key, int32_t *__restrict__ row_oct0,
                              int32_t *__restrict__ row_plane, int32_t *__restrict__ plane_z,
                              int32_t *__restrict__ plane_row0)
{
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r <= half * half) row_oct0[r] = (int32_t)(r * half);
  if (r < half * half) {
    row_key[r] = (uint64_t)(r % half) | ((uint64_t)(r / half) << AHF_KEY_BITS);
    row_plane[r] = (int32_t)(r / half);
  }
  if (r <= half) plane_row0[r] = (int32_t)(r * half);
  if (r < half) plane_z[r] = (int32_t)r;
}

/* ll(): cell = (unsigned long)(L*pos), cells beyond L-1 go to 0
 * (src/libamr_serial/lltools.c:59-65); key = octet-major node index */
__global__ void k_bin_domain(const float *__restrict__ px, const float *__restrict__ py,
                             const float *__restrict__ pz, int64_t n, int64_t L, uint32_t *__restrict__ key,
                             uint32_t *__restrict__ val)
{
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const double dl = (double)L;
  const float pp[3] = {px[p], py[p], pz[p]};
  int64_t c[3];
  for (int d = 0; d < 3; d++) {
    uint64_t v = (uint64_t)(dl * (double)pp[d]);
    if (v > (uint64_t)(L - 1)) v = 0;
    c[d] = (int64_t)v;
  }
  const int64_t half = L / 2;
  const int64_t o = ((c[2] >> 1) * half + (c[1] >> 1)) * half + (c[0] >> 1);
  key[p] = (uint32_t)(8 * o + (c[2] & 1) * 4 + (c[1] & 1) * 2 + (c[0] & 1));
  val[p] = (uint32_t)p;
}

__global__ void k_iota(uint32_t *__restrict__ v, int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = (uint32_t)i;
}

/* CSR start of every node from the sorted keys: first index with key >= m */
__global__ void k_csr_lower_bound(const uint32_t *__restrict__ skey, int64_t n, int64_t nn,
                                  int64_t *__restrict__ p0)
{
  const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m > nn) return;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)skey[mid] < m) lo = mid + 1; else hi = mid;
  }
  p0[m] = lo;
}

/* one thread per octet: its neighbour row and the run links it needs are
 * read once for the 8 children (ahf_presence_mask_oct); imask, when given,
 * receives the octet's interior children as bits (all 27 present) */
__global__ void k_pmask(level_view v, uint32_t *__restrict__ pmask, uint8_t *__restrict__ imask)
{
  const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= v.n_oct) return;
  int32_t nb[27];
#pragma unroll
  for (int i = 0; i < 27; i++) nb[i] = v.nbr[27 * o + i];
  uint8_t lk0[9], lkm[9];
#pragma unroll
  for (int ez = -1; ez <= 1; ez++)
#pragma unroll
    for (int ey = -1; ey <= 1; ey++) {
      const int li = (ez + 1) * 3 + (ey + 1);
      const int32_t a = nb[ahf_e27(0, ey, ez)], b = nb[ahf_e27(-1, ey, ez)];
      lk0[li] = a >= 0 ? v.oct_link[a] : 0;
      lkm[li] = b >= 0 ? v.oct_link[b] : 0;
    }
  const int64_t ox = ahf_kx(v.oct_key[o]), half = v.L / 2;
  uint4 r0, r1;
  r0.x = ahf_presence_mask_oct(nb, lk0, lkm, ox, half, 0);
  r0.y = ahf_presence_mask_oct(nb, lk0, lkm, ox, half, 1);
  r0.z = ahf_presence_mask_oct(nb, lk0, lkm, ox, half, 2);
  r0.w = ahf_presence_mask_oct(nb, lk0, lkm, ox, half, 3);
  r1.x = ahf_presence_mask_oct(nb, lk0, lkm, ox, half, 4);
  r1.y = ahf_presence_mask_oct(nb, lk0, lkm, ox, half, 5);
  r1.z = ahf_presence_mask_oct(nb, lk0, lkm, ox, half, 6);
  r1.w = ahf_presence_mask_oct(nb, lk0, lkm, ox, half, 7);
  uint4 *out = reinterpret_cast<uint4 *>(pmask + 8 * o);
  out[0] = r0;
  out[1] = r1;
  if (imask) {
    const uint32_t pm[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
    uint32_t im = 0;
#pragma unroll
    for (int c = 0; c < 8; c++) im |= (pm[c] == AHF_FULL27) ? 1u << c : 0u;
    imask[o] = (uint8_t)im;
  }
}

/* weight record of every bucket entry (entries [0, *n)): its particle's
 * TSC weights against the entry's own node; and its position record, which
 * the heavy targets and the relinking read */
__global__ void k_prep(level_view v, const int64_t *__restrict__ n_ptr, int64_t n_max,
                       const uint32_t *__restrict__ pnode, const uint32_t *__restrict__ plist,
                       const float *__restrict__ px, const float *__restrict__ py, const float *__restrict__ pz,
                       double m2pd, ahf_w9 *__restrict__ W, ahf_q4 *__restrict__ qp)
{
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n_max || q >= *n_ptr) return;
  const uint32_t p = plist[q];
  const ahf_q4 e = {px[p], py[p], pz[p], 0.0f};
  ahf_w9 w;
  ahf_entry_weights(&v, (int64_t)pnode[q], e.x, e.y, e.z, m2pd, &w);
  W[q] = w;
  qp[q] = e;
}

/* position record of every bucket entry (entries [0, *n)), for the
 * per-source walk of dense levels */
__global__ void k_prep_q(const int64_t *__restrict__ n_ptr, int64_t n_max, const uint32_t *__restrict__ plist,
                       const float *__restrict__ px, const float *__restrict__ py, const float *__restrict__ pz,
                       ahf_q4 *__restrict__ qp)
{
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n_max || q >= *n_ptr) return;
  const uint32_t p = plist[q];
  ahf_q4 e;
  e.x = px[p];
  e.y = py[p];
  e.z = pz[p];
  e.w = 0.0f;
  qp[q] = e;
}


/* Morton order of a full grid of half^3 octets, half a power of two: the
 * i-th octet in Morton order is the one whose interleaved coordinates are i */
__global__ void k_morton_full(int64_t half, uint32_t *__restrict__ tord)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= half * half * half) return;
  const int64_t x = (int64_t)ahf_compact3((uint64_t)i), y = (int64_t)ahf_compact3((uint64_t)i >> 1),
                z = (int64_t)ahf_compact3((uint64_t)i >> 2);
  tord[i] = (uint32_t)((z * half + y) * half + x);
}

/* Morton order of the next level from this one's: a fine octet is a
 * refined node, its Morton code is the coarse octet's followed by the child
 * index cz*4+cy*2+cx, so the fine octets in Morton order are the refined
 * nodes taken octet by octet in Morton order, children in index order.
 * Position k = 8*(rank of the octet in Morton order) + child. */
__global__ void k_morton_next_flags(const uint32_t *__restrict__ tord, const int32_t *__restrict__ node2oct,
                                    int64_t nn, int32_t *__restrict__ flag)
{
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nn) return;
  flag[k] = node2oct[8 * (int64_t)tord[k >> 3] + (k & 7)] >= 0 ? 1 : 0;
}

__global__ void k_morton_next_emit(const uint32_t *__restrict__ tord, const int32_t *__restrict__ node2oct,
                                   int64_t nn, const int32_t *__restrict__ pos, uint32_t *__restrict__ ftord)
{
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nn) return;
  const int32_t o2 = node2oct[8 * (int64_t)tord[k >> 3] + (k & 7)];
  if (o2 >= 0) ftord[pos[k]] = (uint32_t)o2;
}

/* Morton key of every octet, for the target order of the gather */
__global__ void k_morton_keys(level_view v, uint64_t *__restrict__ mk, uint32_t *__restrict__ idx)
{
  const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= v.n_oct) return;
  mk[o] = ahf_morton(v.oct_key[o]);
  idx[o] = (uint32_t)o;
}

#define AHF_XCDS 8
#define AHF_GL_NB 64 /* source nodes around one octet: 4x4x4 */
/* k_gather_light keeps the records of an octet's 4x4x4 neighbourhood as
 * three word arrays (bucket start, entry count, presence mask) at index
 * i + 4j + 18k, octets 72 words apart: the 8 children of 8 octets reading
 * the same relative source then hit 64 distinct banks ({0,1,4,5,18,19,22,23}
 * + 8 * octet modulo 64; the first 32 lanes also cover 32 banks) */
#define AHF_GL_PS 18
#define AHF_GL_OS 72

/* traversal position t of a target's sources -> offset along one axis, for
 * the axis rotation r (0 inside, 1 at X = 0, 2 at X = L-1; ahf_axis_order) */
__device__ __forceinline__ int rot_offset(int i, int r)
{
  const int v = i + r;
  return (v >= 3 ? v - 3 : v) - 1;
}

/* a target with more contributions than this is folded by a workgroup
 * (heavy_targets): fewer fill its wavefronts only once */
#define AHF_HUGE 2048
/* target n of `total` contributions for the heavy kernels: the list's front,
 * or its back (nn entries, one a node) for the huge ones */
__device__ __forceinline__ void heavy_push(uint32_t *__restrict__ heavy, uint32_t *__restrict__ n_heavy, int64_t nn,
                                           int64_t n, uint64_t total)
{
  if (total > AHF_HUGE) heavy[nn - 1 - (int64_t)atomicAdd(n_heavy + 1, 1u)] = (uint32_t)n;
  else heavy[atomicAdd(n_heavy, 1u)] = (uint32_t)n;
}

/*
 * Exact-order density, one lane per target node.
 *
 * Block b is remapped so that each XCD (blocks are dealt to the 8 XCDs in
 * turn) walks one contiguous stretch of the Morton order of the octets
 * (tord); the 8 children of an octet are 8 adjacent lanes.  The 8 lanes of
 * an octet first load the records of the 64 source nodes of the octet's
 * 4x4x4 neighbourhood (bucket start, entry count, presence mask) into LDS.
 * Each lane then marks, in a 27-bit mask in AHF's traversal order, the
 * sources that contribute (present as get_TSCnodes finds them, non-empty),
 * and walks them as one flat sequence of entries: the wavefront runs as long
 * as its longest lane, not as the sum over sources of the longest bucket.
 * Every contribution is two products of the entry's precomputed weights
 * (k_prep) and the FP32 rounding.  Targets with more than kmax
 * contributions are left to k_gather_heavy.
 */
template <bool OFF32>
__global__ void __launch_bounds__(AHF_BLOCK) k_gather_light(level_view v, const uint32_t *__restrict__ tord,
                                                            int64_t per_xcd, const uint32_t *__restrict__ pmask,
                                                            const int64_t *__restrict__ p0,
                                                            const ahf_w9 *__restrict__ W, int descending,
                                                            uint32_t kmax, float *__restrict__ dens,
                                                            uint32_t *__restrict__ heavy,
                                                            uint32_t *__restrict__ n_heavy)
{
  __shared__ uint32_t s_st[AHF_BLOCK / 8 * AHF_GL_OS], s_ct[AHF_BLOCK / 8 * AHF_GL_OS],
      s_pk[AHF_BLOCK / 8 * AHF_GL_OS];
  const int64_t b = blockIdx.x;
  const int64_t t = ((b % AHF_XCDS) * per_xcd + b / AHF_XCDS) * blockDim.x + threadIdx.x;
  const bool active = t < 8 * v.n_oct;
  const int c = threadIdx.x & 7;
  const int nb0 = (threadIdx.x >> 3) * AHF_GL_OS;
  const int64_t o = active ? (int64_t)tord[t >> 3] : 0;
  if (active) {
    const int32_t *nrow = v.nbr + 27 * o;
    for (int m = 0; m < 8; m++) {
      const int u = c * 8 + m;
      const int i = u & 3, j = (u >> 2) & 3, k = u >> 4;
      const int on = nrow[ahf_e27(i == 0 ? -1 : (i == 3), j == 0 ? -1 : (j == 3), k == 0 ? -1 : (k == 3))];
      uint32_t st = 0u, ct = 0u, pk = 0u;
      if (on >= 0) {
        const int64_t sn = 8 * (int64_t)on + (((k + 1) & 1) << 2 | ((j + 1) & 1) << 1 | ((i + 1) & 1));
        const int64_t a = p0[sn];
        st = (uint32_t)a;
        ct = (uint32_t)(p0[sn + 1] - a);
        pk = pmask[sn];
      }
      const int x = nb0 + i + 4 * j + AHF_GL_PS * k;
      s_st[x] = st;
      s_ct[x] = ct;
      s_pk[x] = pk;
    }
  }
  __syncthreads();
  if (!active) return;
  const int cx = c & 1, cy = (c >> 1) & 1, cz = c >> 2;
  /* neighbourhood record of the source at offset (ex,ey,ez): index
   * own + (ez+1)*18 + (ey+1)*4 + (ex+1) with own the target's corner */
  const int rec0 = nb0 + cz * AHF_GL_PS + cy * 4 + cx;
  const int64_t n = 8 * o + c;
  int64_t X, Y, Z;
  ahf_node_xyz(&v, o, c, &X, &Y, &Z);
  const int rx = X == 0 ? 1 : (X == v.L - 1 ? 2 : 0);
  const int ry = Y == 0 ? 1 : (Y == v.L - 1 ? 2 : 0);
  const int rz = Z == 0 ? 1 : (Z == v.L - 1 ? 2 : 0);
  /* per axis, offset+1 of the source at traversal rank 0, 1, 2 as 2-bit
   * fields (identity 0|1<<2|2<<4 inside the box) */
  const uint32_t px = (uint32_t)(rot_offset(0, rx) + 1) | (uint32_t)(rot_offset(1, rx) + 1) << 2 |
                      (uint32_t)(rot_offset(2, rx) + 1) << 4;
  const uint32_t py = (uint32_t)(rot_offset(0, ry) + 1) | (uint32_t)(rot_offset(1, ry) + 1) << 2 |
                      (uint32_t)(rot_offset(2, ry) + 1) << 4;
  const uint32_t pz = (uint32_t)(rot_offset(0, rz) + 1) | (uint32_t)(rot_offset(1, rz) + 1) << 2 |
                      (uint32_t)(rot_offset(2, rz) + 1) << 4;
  /* contributing sources as bits tz*16 + ty*4 + tx of their traversal ranks */
  uint64_t mask = 0;
  uint64_t total = 0;
#pragma unroll 1
  for (int tz = 0; tz < 3; tz++)
#pragma unroll
    for (int ty = 0; ty < 3; ty++)
#pragma unroll
      for (int tx = 0; tx < 3; tx++) {
        const int ez = rot_offset(tz, rz), ey = rot_offset(ty, ry), ex = rot_offset(tx, rx);
        const int x = rec0 + (ez + 1) * AHF_GL_PS + (ey + 1) * 4 + (ex + 1);
        const uint32_t cnt = s_ct[x], pm = s_pk[x];
        if (((pm >> ((1 - ez) * 9 + (1 - ey) * 3 + (1 - ex))) & 1u) && cnt) {
          mask |= 1ull << (tz * 16 + ty * 4 + tx);
          total += cnt;
        }
      }
  if (total > kmax) {
    heavy_push(heavy, n_heavy, 8 * v.n_oct, n, total);
    return;
  }
  const uint32_t step = descending ? 0xFFFFFFFFu : 1u;
  const char *Wb = reinterpret_cast<const char *>(W);
  float d = -1.0f;
  uint32_t rem = 0, q = 0, oz = 0, oy = 0, ox = 0;
  for (uint32_t it = 0; it < (uint32_t)total; it++) {
    if (rem == 0) {
      const int pos = __builtin_ctzll(mask);
      mask &= mask - 1ull;
      const uint32_t ez1 = (pz >> ((pos >> 4) << 1)) & 3u, ey1 = (py >> (((pos >> 2) & 3) << 1)) & 3u,
                     ex1 = (px >> ((pos & 3) << 1)) & 3u;
      const int x = rec0 + (int)(ez1 * AHF_GL_PS + ey1 * 4 + ex1);
      const uint32_t st = s_st[x];
      rem = s_ct[x];
      q = step == 1u ? st : st + rem - 1u;
      /* byte offsets of a[1-ez], wy[1-ey], wx[1-ex] inside a record */
      oz = (2u - ez1) * 8u;
      oy = 24u + (2u - ey1) * 8u;
      ox = 48u + (2u - ex1) * 8u;
    }
    double w;
    if constexpr (OFF32) {
      const uint32_t base = q * (uint32_t)sizeof(ahf_w9);
      w = *reinterpret_cast<const double *>(Wb + (base + oz)) * *reinterpret_cast<const double *>(Wb + (base + oy)) *
          *reinterpret_cast<const double *>(Wb + (base + ox));
    } else {
      const char *rb = Wb + (uint64_t)q * sizeof(ahf_w9);
      w = *reinterpret_cast<const double *>(rb + oz) * *reinterpret_cast<const double *>(rb + oy) *
          *reinterpret_cast<const double *>(rb + ox);
    }
    d = (float)((double)d + w);
    q += step;
    rem--;
  }
  dens[n] = d;
}

/* contribution of one entry record to a target at offset (-ex,-ey,-ez) from
 * its source node, whose centre is (cx,cy,cz) */
__device__ inline double entry_contrib(const ahf_q4 &e, double cx, double cy, double cz, double L, double m2pd,
                                       int ex, int ey, int ez)
{
  return ahf_contrib(m2pd, ahf_pn_sep(e.x, cx, L), ahf_pn_sep(e.y, cy, L), ahf_pn_sep(e.z, cz, L), -ex, -ey, -ez);
}

/* ahf_tsc_w with the offset known at compile time */
template <int D>
__device__ __forceinline__ double tsc_w_c(double s)
{
  if constexpr (D == 0) return 0.75 - s * s;
  else if constexpr (D < 0) return ((0.5 - s) * (0.5 - s)) / 2;
  else return ((0.5 + s) * (0.5 + s)) / 2;
}

template <int EX, int EY, int EZ>
__device__ __forceinline__ double entry_contrib_c(const ahf_q4 &e, double cx, double cy, double cz, double L,
                                                  double m2pd)
{
  return m2pd * tsc_w_c<-EZ>(ahf_pn_sep(e.z, cz, L)) * tsc_w_c<-EY>(ahf_pn_sep(e.y, cy, L)) *
         tsc_w_c<-EX>(ahf_pn_sep(e.x, cx, L));
}

/*
 * Source (EX,EY,EZ) of a target whose 27 neighbours need no periodic wrap:
 * its entries in walk order (step +1, or -1 as a 32-bit wrap), loaded four
 * at a time ahead of the sequential FP32 rounding.  rec points at the
 * target's own node in the octet's 4x4x4 neighbourhood records.
 */
template <int EX, int EY, int EZ>
__device__ __forceinline__ void gather_source_c(float &d, const uint4 *rec, const ahf_q4 *__restrict__ qp,
                                                uint32_t step, double L, double m2pd, const double *cxv,
                                                const double *cyv, const double *czv)
{
  constexpr int OFF = EZ * 16 + EY * 4 + EX;
  constexpr int BIT = (1 - EZ) * 9 + (1 - EY) * 3 + (1 - EX);
  const uint4 r = rec[OFF];
  if (!((r.z >> BIT) & 1u) || r.y == 0) return;
  const double cx = cxv[EX + 1], cy = cyv[EY + 1], cz = czv[EZ + 1];
  const uint32_t cnt = r.y;
  uint32_t q = step == 1u ? r.x : r.x + cnt - 1u;
  uint32_t k = 0;
  for (; k + 4 <= cnt; k += 4) {
    const ahf_q4 e0 = qp[q], e1 = qp[q + step], e2 = qp[q + 2u * step], e3 = qp[q + 3u * step];
    const double w0 = entry_contrib_c<EX, EY, EZ>(e0, cx, cy, cz, L, m2pd);
    const double w1 = entry_contrib_c<EX, EY, EZ>(e1, cx, cy, cz, L, m2pd);
    const double w2 = entry_contrib_c<EX, EY, EZ>(e2, cx, cy, cz, L, m2pd);
    const double w3 = entry_contrib_c<EX, EY, EZ>(e3, cx, cy, cz, L, m2pd);
    d = (float)((double)d + w0);
    d = (float)((double)d + w1);
    d = (float)((double)d + w2);
    d = (float)((double)d + w3);
    q += 4u * step;
  }
  for (; k < cnt; k++, q += step) d = (float)((double)d + entry_contrib_c<EX, EY, EZ>(qp[q], cx, cy, cz, L, m2pd));
}

#define AHF_GS_ROW(EY, EZ)                                                           \
  gather_source_c<-1, EY, EZ>(d, rec, qp, step, L, m2pd, cxv, cyv, czv);            \
  gather_source_c<0, EY, EZ>(d, rec, qp, step, L, m2pd, cxv, cyv, czv);             \
  gather_source_c<1, EY, EZ>(d, rec, qp, step, L, m2pd, cxv, cyv, czv)
#define AHF_GS_PLANE(EZ) \
  AHF_GS_ROW(-1, EZ);    \
  AHF_GS_ROW(0, EZ);     \
  AHF_GS_ROW(1, EZ)

/*
 * Exact-order density for dense levels, one lane per target node, walking
 * the 27 sources one by one over the entries' position records.
 *
 * Block b is remapped so that each XCD (blocks are dealt to the 8 XCDs in
 * turn) walks one contiguous stretch of the Morton order of the octets
 * (tord); the 8 children of an octet are 8 adjacent lanes.  The 8 lanes of
 * an octet first load the records of the 64 source nodes of the octet's
 * 4x4x4 neighbourhood (bucket start, entry count, presence mask) into LDS;
 * every child then counts and gathers its 27 sources from there.  Targets
 * with more than kmax contributions are left to k_gather_heavy.  Targets
 * away from the periodic faces walk their sources in the fixed order
 * z,y,x = -1,0,1 with compile-time offsets; the others follow AHF's rotated
 * order at the faces (ahf_axis_order).
 */
__global__ void __launch_bounds__(AHF_BLOCK) k_gather_src(level_view v, const uint32_t *__restrict__ tord,
                                                            int64_t per_xcd, const uint32_t *__restrict__ pmask,
                                                            const int64_t *__restrict__ p0,
                                                            const ahf_q4 *__restrict__ qp, int descending,
                                                            double m2pd, uint32_t kmax, float *__restrict__ dens,
                                                            uint32_t *__restrict__ heavy,
                                                            uint32_t *__restrict__ n_heavy)
{
  __shared__ uint4 s_rec[AHF_BLOCK / 8 * AHF_GL_NB];
  const int64_t b = blockIdx.x;
  const int64_t t = ((b % AHF_XCDS) * per_xcd + b / AHF_XCDS) * blockDim.x + threadIdx.x;
  const bool active = t < 8 * v.n_oct;
  const int c = threadIdx.x & 7;
  const int nb0 = (threadIdx.x >> 3) * AHF_GL_NB;
  const int64_t o = active ? (int64_t)tord[t >> 3] : 0;
  if (active) {
    const int32_t *nrow = v.nbr + 27 * o;
    for (int m = 0; m < 8; m++) {
      const int u = c * 8 + m;
      const int i = u & 3, j = (u >> 2) & 3, k = u >> 4;
      const int on = nrow[ahf_e27(i == 0 ? -1 : (i == 3), j == 0 ? -1 : (j == 3), k == 0 ? -1 : (k == 3))];
      uint4 r = make_uint4(0u, 0u, 0u, 0u);
      if (on >= 0) {
        const int64_t sn = 8 * (int64_t)on + (((k + 1) & 1) << 2 | ((j + 1) & 1) << 1 | ((i + 1) & 1));
        const int64_t a = p0[sn];
        r.x = (uint32_t)a;
        r.y = (uint32_t)(p0[sn + 1] - a);
        r.z = pmask[sn];
      }
      s_rec[nb0 + u] = r;
    }
  }
  __syncthreads();
  if (!active) return;
  const int cx = c & 1, cy = (c >> 1) & 1, cz = c >> 2;
  /* the target's own node in the neighbourhood: offsets (dx,dy,dz) add
   * dz*16 + dy*4 + dx */
  const uint4 *rec = s_rec + nb0 + (cz + 1) * 16 + (cy + 1) * 4 + (cx + 1);
  const int64_t n = 8 * o + c;
  uint64_t total = 0;
  for (int ez = -1; ez <= 1; ez++)
    for (int ey = -1; ey <= 1; ey++)
      for (int ex = -1; ex <= 1; ex++) {
        const uint4 r = rec[ez * 16 + ey * 4 + ex];
        if ((r.z >> ((1 - ez) * 9 + (1 - ey) * 3 + (1 - ex))) & 1u) total += r.y;
      }
  if (total > kmax) {
    heavy_push(heavy, n_heavy, 8 * v.n_oct, n, total);
    return;
  }
  const double L = (double)v.L;
  int64_t X, Y, Z;
  ahf_node_xyz(&v, o, c, &X, &Y, &Z);
  double cxv[3], cyv[3], czv[3];
  ahf_centres3(X, v.L, cxv);
  ahf_centres3(Y, v.L, cyv);
  ahf_centres3(Z, v.L, czv);
  float d = -1.0f;
  const bool inner = X > 0 && X < v.L - 1 && Y > 0 && Y < v.L - 1 && Z > 0 && Z < v.L - 1;
  if (inner) {
    const uint32_t step = descending ? 0xFFFFFFFFu : 1u;
    AHF_GS_PLANE(-1);
    AHF_GS_PLANE(0);
    AHF_GS_PLANE(1);
  } else {
    int oz[3], oy[3], ox[3];
    ahf_axis_order(Z, v.L, oz);
    ahf_axis_order(Y, v.L, oy);
    ahf_axis_order(X, v.L, ox);
    for (int a3 = 0; a3 < 3; a3++)
      for (int b3 = 0; b3 < 3; b3++)
        for (int e3 = 0; e3 < 3; e3++) {
          const int ez = oz[a3], ey = oy[b3], ex = ox[e3];
          const uint4 r = rec[ez * 16 + ey * 4 + ex];
          if (!((r.z >> ((1 - ez) * 9 + (1 - ey) * 3 + (1 - ex))) & 1u)) continue;
          const int64_t cnt = r.y;
          if (cnt == 0) continue;
          const int64_t q0 = r.x;
          const double scx = cxv[ex + 1], scy = cyv[ey + 1], scz = czv[ez + 1];
          for (int64_t k = 0; k < cnt; k++)
            d = (float)((double)d +
                        entry_contrib(qp[descending ? q0 + cnt - 1 - k : q0 + k], scx, scy, scz, L, m2pd, ex, ey, ez));
        }
  }
  dens[n] = d;
}

#define AHF_SLAB 16                          /* target tile: 16x16 nodes of one plane */
#define AHF_SLAB_W (AHF_SLAB + 2)            /* its sources in one plane: 18x18 nodes */
#define AHF_SLAB_N (AHF_SLAB_W * AHF_SLAB_W)
#define AHF_FULL_CAP_BIG 2752                /* staged entries per plane, dense levels */
#define AHF_FULL_CAP_SMALL 448               /* the same for about one entry per node */

/* node (X,Y,Z) of a level that holds every octet: its octets are all
 * (L/2)^3 keys in (z,y,x) order */
__device__ __forceinline__ int64_t full_node(int64_t X, int64_t Y, int64_t Z, int64_t H)
{
  const int64_t o = ((Z >> 1) * H + (Y >> 1)) * H + (X >> 1);
  return 8 * o + ((Z & 1) << 2 | (Y & 1) << 1 | (X & 1));
}

/* LDS of one workgroup of k_gather_full: bucket start and entry count of
 * three source planes' nodes, the slot offsets and entries of the staged one
 * (FULL: nine weights an entry, else the three separations) */
template <int CAP, bool FULL>
struct FullShared {
  double cx[AHF_SLAB_W], cy[AHF_SLAB_W];
  double e[(FULL ? 9 : 3) * CAP];
  uint32_t start[3 * AHF_SLAB_N], cnt[3 * AHF_SLAB_N], off[AHF_SLAB_N + 1];
  union {
    uint32_t slab_pm[3 * AHF_SLAB_N];
    struct {
      uint32_t pm[AHF_SLAB_N], q[FULL ? 9 * AHF_BLOCK : 1];
    } march;
  };
};

/* ahf_tsc_w(s, d) for an offset d known only at run time, as
 * A + B*(C + D*s)^2 with
 *   d =  0: C = 0,   D = 1,  A = 0.75, B = -1   -> 0.75 - s*s
 *   d = +1: C = 0.5, D = 1,  A = 0,    B = 0.5  -> ((0.5 + s)^2)/2
 *   d = -1: C = 0.5, D = -1, A = 0,    B = 0.5  -> ((0.5 - s)^2)/2
 * Every step is exact or rounds exactly as AHF's formula (products with
 * +-1 and 0.5 and sums with 0 are exact, x + (-y) is x - y), so the bits
 * are those of ahf_tsc_w. */
struct TscRt {
  double A, B, C, D;
  __device__ __forceinline__ explicit TscRt(int d)
      : A(d == 0 ? 0.75 : 0.0), B(d == 0 ? -1.0 : 0.5), C(d == 0 ? 0.0 : 0.5), D(d < 0 ? -1.0 : 1.0)
  {
  }
  __device__ __forceinline__ double operator()(double s) const
  {
    const double q = C + D * s;
    return A + B * (q * q);
  }
};

/*
 * Exact-order density of one 16x16 tile of target nodes of the plane Z of a
 * level that holds every octet, by one workgroup, one lane per target: for
 * the planes Z = 0 and Z = L-1, whose z order wraps (the others march).
 *
 * All targets of the tile share Z, so they visit the three source planes in
 * the same order (ahf_axis_order of Z).  The workgroup stages one source
 * plane at a time: the entries of its 18x18 source nodes are copied into
 * LDS, each as m2pd*wz (wz the TSC weight along z for this plane's offset)
 * and either its separations sy, sx (W9 false) or its three weights along
 * y and along x (W9 true).  Every lane then walks its (up to) nine sources
 * of the plane in AHF's order, each source's entries in list order, and
 * rounds ((m2pd*wz)*wy)*wx into its FP32 node value as AHF does.  Entries of
 * nodes that do not fit in the CAP staged slots are read from the position
 * records instead, with the same arithmetic.  Targets with more than kmax
 * contributions are left to k_gather_heavy.
 */
template <int CAP, bool W9>
__device__ __forceinline__ void gather_slab(const level_view &v, int64_t tx, int64_t ty, int64_t Z, FullShared<CAP, W9> &S,
                                            const uint32_t *__restrict__ pmask, const int64_t *__restrict__ p0,
                                            const ahf_q4 *__restrict__ qp, int descending, double m2pd, uint32_t kmax,
                                            float *__restrict__ dens, uint32_t *__restrict__ heavy,
                                            uint32_t *__restrict__ n_heavy)
{
  uint32_t *const s_start = S.start, *const s_cnt = S.cnt, *const s_pm = S.slab_pm, *const s_off = S.off;
  double *const s_cx = S.cx, *const s_cy = S.cy, *const s_e = S.e;
  const int64_t L = v.L, H = L >> 1;
  const int tid = threadIdx.x, lx = tid & (AHF_SLAB - 1), ly = tid / AHF_SLAB;
  const int64_t X = tx * AHF_SLAB + lx, Y = ty * AHF_SLAB + ly;
  const double Ld = (double)L;
  int oz[3], oy[3], ox[3];
  ahf_axis_order(Z, L, oz);
  ahf_axis_order(Y, L, oy);
  ahf_axis_order(X, L, ox);
  /* bucket start, entry count and presence mask of the 3 x 18 x 18 source
   * nodes, planes in traversal order; centres of the 18 source columns and
   * rows */
  for (int i = tid; i < 3 * AHF_SLAB_N; i += AHF_BLOCK) {
    const int k = i / AHF_SLAB_N, u = i - k * AHF_SLAB_N;
    const int64_t Xs = ahf_wrap(tx * AHF_SLAB - 1 + u % AHF_SLAB_W, L);
    const int64_t Ys = ahf_wrap(ty * AHF_SLAB - 1 + u / AHF_SLAB_W, L);
    const int64_t sn = full_node(Xs, Ys, ahf_wrap(Z + oz[k], L), H);
    const int64_t a = p0[sn];
    s_start[i] = (uint32_t)a;
    s_cnt[i] = (uint32_t)(p0[sn + 1] - a);
    s_pm[i] = pmask[sn];
  }
  if (tid < AHF_SLAB_W) s_cx[tid] = ahf_centre(ahf_wrap(tx * AHF_SLAB - 1 + tid, L), Ld);
  else if (tid < 2 * AHF_SLAB_W)
    s_cy[tid - AHF_SLAB_W] = ahf_centre(ahf_wrap(ty * AHF_SLAB - 1 + (tid - AHF_SLAB_W), L), Ld);
  __syncthreads();
  /* contributing sources as bits k*9 + ty*3 + tx of their traversal ranks */
  uint32_t mask = 0;
  uint64_t total = 0;
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int bb = 0; bb < 3; bb++)
#pragma unroll
      for (int e = 0; e < 3; e++) {
        const int ez = oz[k], ey = oy[bb], ex = ox[e];
        const int u = k * AHF_SLAB_N + (ly + 1 + ey) * AHF_SLAB_W + (lx + 1 + ex);
        if (!((s_pm[u] >> ((1 - ez) * 9 + (1 - ey) * 3 + (1 - ex))) & 1u)) continue;
        total += s_cnt[u];
        if (s_cnt[u]) mask |= 1u << (k * 9 + bb * 3 + e);
      }
  const int64_t n = full_node(X, Y, Z, H);
  const bool inside = X < L && Y < L; /* the last tile of a row or column may be partial */
  const bool active = inside && total <= kmax;
  if (inside && !active) heavy_push(heavy, n_heavy, 8 * v.n_oct, n, total);
  const uint32_t step = descending ? 0xFFFFFFFFu : 1u;
  float d = -1.0f;
  for (int k = 0; k < 3; k++) {
    const int ez = oz[k];
    const uint32_t *cnt_k = s_cnt + k * AHF_SLAB_N;
    const uint32_t *start_k = s_start + k * AHF_SLAB_N;
    /* LDS slot of each node's first entry: node pairs per thread */
    uint32_t c0 = 0, c1 = 0;
    if (tid < AHF_SLAB_N / 2) {
      c0 = cnt_k[2 * tid];
      c1 = cnt_k[2 * tid + 1];
    }
    uint32_t tot = 0;
    const uint32_t ex0 = ahf::block_excl_scan<uint32_t>(c0 + c1, &tot);
    if (tid < AHF_SLAB_N / 2) {
      s_off[2 * tid] = ex0;
      s_off[2 * tid + 1] = ex0 + c0;
    }
    if (tid == 0) s_off[AHF_SLAB_N] = tot;
    __syncthreads();
    const double czs = ahf_centre(ahf_wrap(Z + ez, L), Ld);
    const TscRt tz(-ez);
    const uint32_t lim = tot < (uint32_t)CAP ? tot : (uint32_t)CAP;
    for (uint32_t e = tid; e < lim; e += AHF_BLOCK) {
      /* the node holding entry e: s_off[lo] <= e < s_off[lo + 1] */
      int lo = 0, hi = AHF_SLAB_N;
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (s_off[mid] <= e) lo = mid;
        else hi = mid;
      }
      if (s_off[lo] + cnt_k[lo] > (uint32_t)CAP) continue; /* read from the records */
      const ahf_q4 q = qp[start_k[lo] + (e - s_off[lo])];
      const int row = lo / AHF_SLAB_W, col = lo - row * AHF_SLAB_W;
      const double sx = ahf_pn_sep(q.x, s_cx[col], Ld);
      const double sy = ahf_pn_sep(q.y, s_cy[row], Ld);
      s_e[e] = m2pd * tz(ahf_pn_sep(q.z, czs, Ld));
      if constexpr (W9) {
        s_e[1 * CAP + e] = tsc_w_c<-1>(sy);
        s_e[2 * CAP + e] = tsc_w_c<0>(sy);
        s_e[3 * CAP + e] = tsc_w_c<1>(sy);
        s_e[4 * CAP + e] = tsc_w_c<-1>(sx);
        s_e[5 * CAP + e] = tsc_w_c<0>(sx);
        s_e[6 * CAP + e] = tsc_w_c<1>(sx);
      } else {
        s_e[CAP + e] = sy;
        s_e[2 * CAP + e] = sx;
      }
    }
    __syncthreads();
    if (active) {
      const uint32_t m9 = (mask >> (9 * k)) & 0x1FFu;
#pragma unroll
      for (int t = 0; t < 9; t++) {
        if (!((m9 >> t) & 1u)) continue;
        const int ey = oy[t / 3], ex = ox[t % 3];
        const int u = (ly + 1 + ey) * AHF_SLAB_W + (lx + 1 + ex);
        const uint32_t cnt = cnt_k[u], o = s_off[u];
        if (o + cnt <= (uint32_t)CAP) {
          uint32_t q = descending ? o + cnt - 1u : o;
          if constexpr (W9) {
            /* weight index 1 - e for a source at offset e */
            const double *wy = s_e + (2 - ey) * CAP;
            const double *wx = s_e + (5 - ex) * CAP;
            for (uint32_t j = 0; j < cnt; j++, q += step) d = (float)((double)d + (s_e[q] * wy[q]) * wx[q]);
          } else {
            const TscRt fy(-ey), fx(-ex);
            for (uint32_t j = 0; j < cnt; j++, q += step)
              d = (float)((double)d + (s_e[q] * fy(s_e[CAP + q])) * fx(s_e[2 * CAP + q]));
          }
        } else {
          const TscRt fy(-ey), fx(-ex);
          const double cxs = s_cx[lx + 1 + ex], cys = s_cy[ly + 1 + ey];
          uint32_t q = descending ? start_k[u] + cnt - 1u : start_k[u];
          for (uint32_t j = 0; j < cnt; j++, q += step) {
            const ahf_q4 r = qp[q];
            const double az = m2pd * tz(ahf_pn_sep(r.z, czs, Ld));
            d = (float)((double)d + (az * fy(ahf_pn_sep(r.y, cys, Ld))) * fx(ahf_pn_sep(r.x, cxs, Ld)));
          }
        }
      }
    }
    __syncthreads();
  }
  if (active) dens[n] = d;
}

/* shared state of one marching workgroup (gather_march) */
struct MarchView {
  const uint32_t *cnt, *start, *off; /* the walked plane's slot */
  const double *e;                   /* its staged entries */
  const double *cx, *cy;             /* source column and row centres */
  const ahf_q4 *qp;
  double m2pd, L, czs;
  uint32_t step;
  int lx, ly;
};

/* the contribution of a staged or recorded entry to the three targets above,
 * at and below the walked plane, in the FP32 values d0 (plane P+1, which sees
 * the source at z offset -1), d1 (plane P) and d2 (plane P-1), each only
 * where its use flag is set */
__device__ __forceinline__ void fold3(float &d0, float &d1, float &d2, bool u0, bool u1, bool u2, double a0, double a1,
                                      double a2, double wy, double wx)
{
  const float n0 = (float)((double)d0 + (a0 * wy) * wx);
  const float n1 = (float)((double)d1 + (a1 * wy) * wx);
  const float n2 = (float)((double)d2 + (a2 * wy) * wx);
  d0 = u0 ? n0 : d0;
  d1 = u1 ? n1 : d1;
  d2 = u2 ? n2 : d2;
}

/*
 * Source (B,E) (traversal ranks along y and x) of the walked plane for the
 * lane's three targets.  Inside the box (FACE false) the offsets are B-1,
 * E-1 and the TSC weights take compile-time forms; at the periodic faces
 * they follow the lane's rotated order.  The z weights of the three targets
 * are those of offsets -1, 0, +1 (TSC index d = 1, 0, -1).
 */
template <int CAP, bool FULL, bool FACE, int B, int E>
__device__ __forceinline__ void march_source(const MarchView &m, const int *oy, const int *ox, uint32_t m0, uint32_t m1,
                                             uint32_t m2, float &d0, float &d1, float &d2)
{
  constexpr int BIT = B * 3 + E;
  const bool u0 = (m0 >> BIT) & 1u, u1 = (m1 >> BIT) & 1u, u2 = (m2 >> BIT) & 1u;
  if (!(u0 || u1 || u2)) return;
  const int ey = FACE ? oy[B] : B - 1, ex = FACE ? ox[E] : E - 1;
  const int u = (m.ly + 1 + ey) * AHF_SLAB_W + (m.lx + 1 + ex);
  const uint32_t cnt = m.cnt[u], o = m.off[u];
  const TscRt fy(-ey), fx(-ex);
  if (o + cnt <= (uint32_t)CAP) {
    uint32_t q = m.step == 1u ? o : o + cnt - 1u;
    for (uint32_t j = 0; j < cnt; j++, q += m.step) {
      double a0, a1, a2, wy, wx;
      if constexpr (FULL) {
        a0 = m.e[q];
        a1 = m.e[CAP + q];
        a2 = m.e[2 * CAP + q];
        wy = m.e[(4 - ey) * CAP + q];
        wx = m.e[(7 - ex) * CAP + q];
      } else {
        const double sz = m.e[q], sy = m.e[CAP + q], sx = m.e[2 * CAP + q];
        a0 = m.m2pd * tsc_w_c<1>(sz);
        a1 = m.m2pd * tsc_w_c<0>(sz);
        a2 = m.m2pd * tsc_w_c<-1>(sz);
        if constexpr (FACE) {
          wy = fy(sy);
          wx = fx(sx);
        } else {
          wy = tsc_w_c<1 - B>(sy);
          wx = tsc_w_c<1 - E>(sx);
        }
      }
      fold3(d0, d1, d2, u0, u1, u2, a0, a1, a2, wy, wx);
    }
  } else {
    const double cxs = m.cx[m.lx + 1 + ex], cys = m.cy[m.ly + 1 + ey];
    uint32_t q = m.step == 1u ? m.start[u] : m.start[u] + cnt - 1u;
    for (uint32_t j = 0; j < cnt; j++, q += m.step) {
      const ahf_q4 r = m.qp[q];
      const double sz = ahf_pn_sep(r.z, m.czs, m.L);
      fold3(d0, d1, d2, u0, u1, u2, m.m2pd * tsc_w_c<1>(sz), m.m2pd * tsc_w_c<0>(sz), m.m2pd * tsc_w_c<-1>(sz),
            fy(ahf_pn_sep(r.y, cys, m.L)), fx(ahf_pn_sep(r.x, cxs, m.L)));
    }
  }
}

template <int CAP, bool FULL, bool FACE>
__device__ __forceinline__ void march_plane(const MarchView &m, const int *oy, const int *ox, uint32_t m0, uint32_t m1,
                                            uint32_t m2, float &d0, float &d1, float &d2)
{
  march_source<CAP, FULL, FACE, 0, 0>(m, oy, ox, m0, m1, m2, d0, d1, d2);
  march_source<CAP, FULL, FACE, 0, 1>(m, oy, ox, m0, m1, m2, d0, d1, d2);
  march_source<CAP, FULL, FACE, 0, 2>(m, oy, ox, m0, m1, m2, d0, d1, d2);
  march_source<CAP, FULL, FACE, 1, 0>(m, oy, ox, m0, m1, m2, d0, d1, d2);
  march_source<CAP, FULL, FACE, 1, 1>(m, oy, ox, m0, m1, m2, d0, d1, d2);
  march_source<CAP, FULL, FACE, 1, 2>(m, oy, ox, m0, m1, m2, d0, d1, d2);
  march_source<CAP, FULL, FACE, 2, 0>(m, oy, ox, m0, m1, m2, d0, d1, d2);
  march_source<CAP, FULL, FACE, 2, 1>(m, oy, ox, m0, m1, m2, d0, d1, d2);
  march_source<CAP, FULL, FACE, 2, 2>(m, oy, ox, m0, m1, m2, d0, d1, d2);
}

/* presence and entry counts of a lane's nine sources in one staged source
 * plane S, for the three targets that visit it: role 0 is the target S+1
 * (S is its z offset -1), role 1 the target S, role 2 the target S-1.
 * Bit r*9 + B*3 + E of m is set when the source at traversal ranks (B,E)
 * is present for role r (get_TSCnodes) and holds entries; c[r] sums them. */
struct PlaneSum {
  uint32_t m, c0, c1, c2;
};

__device__ __forceinline__ PlaneSum plane_sum(const uint32_t *cnt, const uint32_t *pm, const int *oy, const int *ox,
                                              int lx, int ly)
{
  PlaneSum r = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int bb = 0; bb < 3; bb++)
#pragma unroll
    for (int e = 0; e < 3; e++) {
      const int ey = oy[bb], ex = ox[e];
      const int u = (ly + 1 + ey) * AHF_SLAB_W + (lx + 1 + ex);
      const uint32_t c = cnt[u];
      if (!c) continue;
      const uint32_t w = pm[u] >> ((1 - ey) * 3 + (1 - ex));
      const int t = bb * 3 + e;
      /* role r sees the plane at z offset r-1: presence bit (2-r)*9 + ... */
      if ((w >> 18) & 1u) {
        r.m |= 1u << t;
        r.c0 += c;
      }
      if ((w >> 9) & 1u) {
        r.m |= 1u << (9 + t);
        r.c1 += c;
      }
      if (w & 1u) {
        r.m |= 1u << (18 + t);
        r.c2 += c;
      }
    }
  return r;
}

/*
 * Exact-order density of the planes 1 <= Z <= L-2 of a level that holds
 * every octet, whose sources lie in the planes Z-1, Z, Z+1 in that order.
 * One workgroup per 16x16 column tile and run of zn target planes, one lane
 * per (x,y) column.  The workgroup marches up through the source planes,
 * staging each one in LDS once (as in gather_slab), and every lane folds
 * the staged plane P into its three open targets: plane P+1 (its first
 * source plane), P (its second) and P-1 (its third, after which the value
 * is final).  All three visit the plane's sources in the same order, so one
 * walk serves them and the TSC weights along y and x are shared.  Bucket
 * records of the planes P, P+1, P+2 are kept in a ring of three slots, and
 * each lane summarises a plane's sources once when it arrives, so that
 * target P+1's contribution count (for the kmax test) is known when it
 * opens.  FULL stages the nine weights of each entry and walks the plane's
 * sources as one flat sequence from a per-lane queue in LDS (few entries
 * per source: the wavefront runs as long as its longest lane over the
 * plane, not over each source); otherwise the separations are staged and
 * the sources are walked one by one with compile-time weights.
 */
template <int CAP, bool FULL>
__device__ __forceinline__ void gather_march(const level_view &v, int64_t tx, int64_t ty, int64_t T, int64_t ch, int64_t zn,
                                             FullShared<CAP, FULL> &S, const uint32_t *__restrict__ pmask,
                                             const int64_t *__restrict__ p0, const ahf_q4 *__restrict__ qp,
                                             int descending, double m2pd, uint32_t kmax, float *__restrict__ dens,
                                             uint32_t *__restrict__ heavy, uint32_t *__restrict__ n_heavy)
{
  uint32_t *const s_start = S.start, *const s_cnt = S.cnt, *const s_pm = S.march.pm, *const s_off = S.off,
                  *const s_q = S.march.q;
  double *const s_cx = S.cx, *const s_cy = S.cy, *const s_e = S.e;
  const int64_t L = v.L, H = L >> 1;
  const int64_t Z0 = 1 + ch * zn, Z1 = Z0 + zn < L - 1 ? Z0 + zn : L - 1;
  const int tid = threadIdx.x, lx = tid & (AHF_SLAB - 1), ly = tid / AHF_SLAB;
  const int64_t X = tx * AHF_SLAB + lx, Y = ty * AHF_SLAB + ly;
  const double Ld = (double)L;
  const bool face = tx == 0 || tx == T - 1 || ty == 0 || ty == T - 1;
  const bool inside = X < L && Y < L; /* the last tile of a row or column may be partial */
  int oy[3], ox[3];
  ahf_axis_order(Y, L, oy);
  ahf_axis_order(X, L, ox);
  if (tid < AHF_SLAB_W) s_cx[tid] = ahf_centre(ahf_wrap(tx * AHF_SLAB - 1 + tid, L), Ld);
  else if (tid < 2 * AHF_SLAB_W)
    s_cy[tid - AHF_SLAB_W] = ahf_centre(ahf_wrap(ty * AHF_SLAB - 1 + (tid - AHF_SLAB_W), L), Ld);
  /* bucket records of source plane Zs into ring slot Zs mod 3 (presence
   * masks into the one slot that plane_sum reads) */
  auto load_plane = [&](int64_t Zs) {
    const int slot = (int)(Zs % 3);
    const int64_t Zw = ahf_wrap(Zs, L);
    for (int i = tid; i < AHF_SLAB_N; i += AHF_BLOCK) {
      const int64_t Xs = ahf_wrap(tx * AHF_SLAB - 1 + i % AHF_SLAB_W, L);
      const int64_t Ys = ahf_wrap(ty * AHF_SLAB - 1 + i / AHF_SLAB_W, L);
      const int64_t sn = full_node(Xs, Ys, Zw, H);
      const int64_t a = p0[sn];
      s_start[slot * AHF_SLAB_N + i] = (uint32_t)a;
      s_cnt[slot * AHF_SLAB_N + i] = (uint32_t)(p0[sn + 1] - a);
      s_pm[i] = pmask[sn]; /* summarised before the next load */
    }
  };
  auto sum_of = [&](int64_t Zs) {
    const int slot = (int)(Zs % 3);
    return plane_sum(s_cnt + slot * AHF_SLAB_N, s_pm, oy, ox, lx, ly);
  };
  load_plane(Z0 - 1);
  __syncthreads();
  PlaneSum sP = sum_of(Z0 - 1);
  __syncthreads();
  load_plane(Z0);
  __syncthreads();
  PlaneSum sP1 = sum_of(Z0);
  __syncthreads();
  MarchView m;
  m.off = s_off;
  m.e = s_e;
  m.cx = s_cx;
  m.cy = s_cy;
  m.qp = qp;
  m.m2pd = m2pd;
  m.L = Ld;
  m.step = descending ? 0xFFFFFFFFu : 1u;
  m.lx = lx;
  m.ly = ly;
  /* the open targets: P+1 (n), P (c), P-1 (p); plane summaries of P, P+1 */
  float dn = -1.0f, dc = -1.0f, dp = -1.0f;
  uint32_t mn = 0, mc = 0, mp = 0;
  bool an = false, ac = false, ap = false;
  for (int64_t P = Z0 - 1; P <= Z1; P++) {
    load_plane(P + 2);
    __syncthreads();
    const PlaneSum sP2 = sum_of(P + 2);
    const int sp = (int)(P % 3);
    const uint32_t *cnt_p = s_cnt + sp * AHF_SLAB_N, *start_p = s_start + sp * AHF_SLAB_N;
    uint32_t c0 = 0, c1 = 0;
    if (tid < AHF_SLAB_N / 2) {
      c0 = cnt_p[2 * tid];
      c1 = cnt_p[2 * tid + 1];
    }
    uint32_t tot = 0;
    const uint32_t ex0 = ahf::block_excl_scan<uint32_t>(c0 + c1, &tot);
    if (tid < AHF_SLAB_N / 2) {
      s_off[2 * tid] = ex0;
      s_off[2 * tid + 1] = ex0 + c0;
    }
    if (tid == 0) s_off[AHF_SLAB_N] = tot;
    __syncthreads();
    const double czs = ahf_centre(ahf_wrap(P, L), Ld);
    if constexpr (FULL) {
      /* one thread per staged entry (the node holding entry e found by a
       * binary search of the offsets): the plane's work spread evenly,
       * whatever the nodes' counts */
      const uint32_t lim = tot < (uint32_t)CAP ? tot : (uint32_t)CAP;
      for (uint32_t e = tid; e < lim; e += AHF_BLOCK) {
        int lo = 0, hi = AHF_SLAB_N;
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (s_off[mid] <= e) lo = mid;
          else hi = mid;
        }
        const int u = lo;
        if (s_off[u] + cnt_p[u] > (uint32_t)CAP) continue; /* read from the records */
        const int row = u / AHF_SLAB_W, col = u - row * AHF_SLAB_W;
        const double cxs = s_cx[col], cys = s_cy[row];
        {
          const ahf_q4 q = qp[start_p[u] + (e - s_off[u])];
          const double sz = ahf_pn_sep(q.z, czs, Ld);
          const double sy = ahf_pn_sep(q.y, cys, Ld);
          const double sx = ahf_pn_sep(q.x, cxs, Ld);
          s_e[e] = m2pd * tsc_w_c<1>(sz);
          s_e[CAP + e] = m2pd * tsc_w_c<0>(sz);
          s_e[2 * CAP + e] = m2pd * tsc_w_c<-1>(sz);
          s_e[3 * CAP + e] = tsc_w_c<-1>(sy);
          s_e[4 * CAP + e] = tsc_w_c<0>(sy);
          s_e[5 * CAP + e] = tsc_w_c<1>(sy);
          s_e[6 * CAP + e] = tsc_w_c<-1>(sx);
          s_e[7 * CAP + e] = tsc_w_c<0>(sx);
          s_e[8 * CAP + e] = tsc_w_c<1>(sx);
        }
      }
    } else {
      const uint32_t lim = tot < (uint32_t)CAP ? tot : (uint32_t)CAP;
      for (uint32_t e = tid; e < lim; e += AHF_BLOCK) {
        /* the node holding entry e: s_off[lo] <= e < s_off[lo + 1] */
        int lo = 0, hi = AHF_SLAB_N;
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (s_off[mid] <= e) lo = mid;
          else hi = mid;
        }
        if (s_off[lo] + cnt_p[lo] > (uint32_t)CAP) continue; /* read from the records */
        const ahf_q4 q = qp[start_p[lo] + (e - s_off[lo])];
        const int row = lo / AHF_SLAB_W, col = lo - row * AHF_SLAB_W;
        s_e[e] = ahf_pn_sep(q.z, czs, Ld);
        s_e[CAP + e] = ahf_pn_sep(q.y, s_cy[row], Ld);
        s_e[2 * CAP + e] = ahf_pn_sep(q.x, s_cx[col], Ld);
      }
    }
    /* target P+1 opens: planes P (its z offset -1), P+1 (0), P+2 (+1) */
    mn = 0;
    an = false;
    dn = -1.0f;
    if (inside && P + 1 >= Z0 && P + 1 < Z1) {
      const uint64_t total = (uint64_t)sP.c0 + sP1.c1 + sP2.c2;
      an = total <= kmax;
      if (an) mn = (sP.m & 0x1FFu) | (sP1.m & (0x1FFu << 9)) | (sP2.m & (0x1FFu << 18));
      else heavy_push(heavy, n_heavy, 8 * v.n_oct, full_node(X, Y, P + 1, H), total);
    }
    __syncthreads();
    m.cnt = cnt_p;
    m.start = start_p;
    m.czs = czs;
    /* plane P is the first source plane of P+1, the second of P, the third of P-1 */
    const uint32_t m0 = mn & 0x1FFu, m1 = ac ? (mc >> 9) & 0x1FFu : 0u, m2 = ap ? (mp >> 18) & 0x1FFu : 0u;
    if constexpr (FULL) {
      /* Rows fast path (ascending lists, every source staged): the three
       * sources of one source row are adjacent nodes of the staged plane, so
       * their entries form one range of the staged order, walked from the
       * first source in the lane's x order and wrapping round the range
       * (the order at the periodic faces is a rotation); the source of an
       * entry, and so its x weight, follows from the range's inner
       * boundaries.  A lane qualifies when each of its three targets takes
       * either none or all of the plane's non-empty sources, and the
       * wavefront takes the path only if all its lanes qualify. */
      bool rows = false;
      const int rot = ox[0] + 1; /* first source in x order: 0, 1 or 2 along a row */
      if (tot <= (uint32_t)CAP && m.step == 1u) {
        uint32_t ne9 = 0;
#pragma unroll
        for (int bb = 0; bb < 3; bb++) {
          const int u = (ly + 1 + oy[bb]) * AHF_SLAB_W + lx;
          const uint32_t o0 = s_off[u], o1 = s_off[u + 1], o2 = s_off[u + 2], o3 = s_off[u + 3];
#pragma unroll
          for (int e = 0; e < 3; e++) {
            const int ex = ox[e];
            const uint32_t ce = ex < 0 ? o1 - o0 : (ex == 0 ? o2 - o1 : o3 - o2);
            if (ce) ne9 |= 1u << (bb * 3 + e);
          }
        }
        const bool ok = (m0 == 0u || m0 == ne9) && (m1 == 0u || m1 == ne9) && (m2 == 0u || m2 == ne9);
        rows = __ballot(!ok) == 0ull;
      }
      if (rows) {
        const bool r0 = m0 != 0u, r1 = m1 != 0u, r2 = m2 != 0u;
        const int oy0 = oy[0], oy1 = oy[1], oy2 = oy[2];
        uint32_t ntot = 0;
        if (r0 || r1 || r2) {
#pragma unroll
          for (int bb = 0; bb < 3; bb++) {
            const int u = (ly + 1 + oy[bb]) * AHF_SLAB_W + lx;
            ntot += s_off[u + 3] - s_off[u];
          }
        }
        /* the current row: next entry q, entries left, range [lo, hi) with
         * inner boundaries b1, b2, and the offset of its y weight */
        uint32_t q = 0, rem = 0, lo = 0, hi = 0, b1 = 0, b2 = 0, y3 = 0;
        int br = -1;
        for (uint32_t it = 0; it < ntot; it++) {
          while (rem == 0u) {
            br++;
            const int ey = br == 0 ? oy0 : (br == 1 ? oy1 : oy2);
            const int u = (ly + 1 + ey) * AHF_SLAB_W + lx;
            lo = s_off[u];
            b1 = s_off[u + 1];
            b2 = s_off[u + 2];
            hi = s_off[u + 3];
            rem = hi - lo;
            q = ahf_row_start(lo, b1, b2, hi, rot);
            y3 = (3u + (uint32_t)(1 - ey)) * (uint32_t)CAP;
          }
          /* x weight index 1 - ex of the entry's source: 8, 7, 6 along the row */
          const uint32_t wx = (8u - ahf_row_src(q, b1, b2)) * (uint32_t)CAP;
          fold3(dn, dc, dp, r0, r1, r2, s_e[q], s_e[CAP + q], s_e[2 * CAP + q], s_e[y3 + q], s_e[wx + q]);
          q = ahf_row_next(q, lo, hi);
          rem--;
        }
      } else {
      /* the lane's sources of this plane in order, as one flat sequence */
      uint32_t *qq = s_q + tid * 9;
      if (tot <= (uint32_t)CAP) {
        /* every source of the plane is staged (the common case): LDS slot
         * (10 bits), count (12 bits; a light target's sources hold at most
         * kmax < 4096 entries), roles (3), weight indices 1-ey and 1-ex;
         * the next source's word is read one switch ahead */
        uint32_t nq = 0, ntot = 0;
#pragma unroll
        for (int t = 0; t < 9; t++) {
          const uint32_t roles = ((m0 >> t) & 1u) | ((m1 >> t) & 1u) << 1 | ((m2 >> t) & 1u) << 2;
          if (!roles) continue;
          const int ey = oy[t / 3], ex = ox[t % 3];
          const int u = (ly + 1 + ey) * AHF_SLAB_W + (lx + 1 + ex);
          const uint32_t c = cnt_p[u];
          qq[nq++] = s_off[u] | c << 10 | roles << 22 | (uint32_t)(1 - ey) << 25 | (uint32_t)(1 - ex) << 27;
          ntot += c;
        }
        uint32_t k = 0, rem = 0, q = 0, nxt = qq[0];
        uint32_t oy3 = 0, ox3 = 0;
        bool r0 = false, r1 = false, r2 = false;
        for (uint32_t it = 0; it < ntot; it++) {
          if (rem == 0) {
            const uint32_t wq = nxt;
            k++;
            nxt = qq[k < 9u ? k : 8u];
            rem = (wq >> 10) & 0xFFFu;
            q = m.step == 1u ? (wq & 0x3FFu) : (wq & 0x3FFu) + rem - 1u;
            r0 = (wq >> 22) & 1u;
            r1 = (wq >> 23) & 1u;
            r2 = (wq >> 24) & 1u;
            oy3 = (3u + ((wq >> 25) & 3u)) * (uint32_t)CAP;
            ox3 = (6u + ((wq >> 27) & 3u)) * (uint32_t)CAP;
          }
          fold3(dn, dc, dp, r0, r1, r2, s_e[q], s_e[CAP + q], s_e[2 * CAP + q], s_e[oy3 + q], s_e[ox3 + q]);
          q += m.step;
          rem--;
        }
      } else {
      uint32_t nq = 0, ntot = 0;
#pragma unroll
      for (int t = 0; t < 9; t++) {
        const uint32_t roles = ((m0 >> t) & 1u) | ((m1 >> t) & 1u) << 1 | ((m2 >> t) & 1u) << 2;
        if (!roles) continue;
        const int ey = oy[t / 3], ex = ox[t % 3];
        const uint32_t u = (uint32_t)((ly + 1 + ey) * AHF_SLAB_W + (lx + 1 + ex));
        const uint32_t c = cnt_p[u], o = s_off[u];
        const uint32_t staged = o + c <= (uint32_t)CAP;
        /* LDS slot or node (10 bits), count (12), roles (3), weight indices
         * 1-ey and 1-ex (2 + 2), staged (1) */
        qq[nq++] = (staged ? o : u) | c << 10 | roles << 22 | (uint32_t)(1 - ey) << 25 | (uint32_t)(1 - ex) << 27 |
                   staged << 29;
        ntot += c;
      }
      uint32_t k = 0, rem = 0, q = 0;
      int iy = 0, ix = 0;
      bool r0 = false, r1 = false, r2 = false, stg = true;
      double cys = 0.0, cxs = 0.0;
      for (uint32_t it = 0; it < ntot; it++) {
        if (rem == 0) {
          const uint32_t wq = qq[k++];
          rem = (wq >> 10) & 0xFFFu;
          r0 = (wq >> 22) & 1u;
          r1 = (wq >> 23) & 1u;
          r2 = (wq >> 24) & 1u;
          iy = (int)((wq >> 25) & 3u);
          ix = (int)((wq >> 27) & 3u);
          stg = (wq >> 29) & 1u;
          const uint32_t first = stg ? (wq & 0x3FFu) : start_p[wq & 0x3FFu];
          q = m.step == 1u ? first : first + rem - 1u;
          if (!stg) {
            cys = s_cy[ly + 2 - iy];
            cxs = s_cx[lx + 2 - ix];
          }
        }
        if (stg) {
          fold3(dn, dc, dp, r0, r1, r2, s_e[q], s_e[CAP + q], s_e[2 * CAP + q], s_e[(3 + iy) * CAP + q],
                s_e[(6 + ix) * CAP + q]);
        } else {
          const ahf_q4 r = qp[q];
          const double sz = ahf_pn_sep(r.z, czs, Ld);
          fold3(dn, dc, dp, r0, r1, r2, m2pd * tsc_w_c<1>(sz), m2pd * tsc_w_c<0>(sz), m2pd * tsc_w_c<-1>(sz),
                TscRt(iy - 1)(ahf_pn_sep(r.y, cys, Ld)), TscRt(ix - 1)(ahf_pn_sep(r.x, cxs, Ld)));
        }
        q += m.step;
        rem--;
      }
      }
      }
    } else {
      if (face) march_plane<CAP, FULL, true>(m, oy, ox, m0, m1, m2, dn, dc, dp);
      else march_plane<CAP, FULL, false>(m, oy, ox, m0, m1, m2, dn, dc, dp);
    }
    if (ap) dens[full_node(X, Y, P - 1, H)] = dp;
    dp = dc;
    dc = dn;
    mp = mc;
    mc = mn;
    ap = ac;
    ac = an;
    sP = sP1;
    sP1 = sP2;
    __syncthreads();
  }
}

/*
 * Exact-order density of a level that holds every octet, L >= AHF_SLAB, in
 * one launch: workgroups [0, nface) take the tiles of the two face planes
 * Z = 0 and L-1 (gather_slab), which would otherwise follow the march alone
 * on the chip (0.29 ms of a 128^3 level's 0.60), the others the column tiles
 * and runs of zn planes between them (gather_march).  Dealt so that each XCD
 * walks a contiguous run of either kind (per_f and per_m workgroups an XCD).
 */
template <int CAP, bool FULL>
__global__ void __launch_bounds__(AHF_BLOCK) k_gather_full(level_view v, int64_t per_f, int64_t per_m, int64_t zn,
                                                           const uint32_t *__restrict__ pmask,
                                                           const int64_t *__restrict__ p0,
                                                           const ahf_q4 *__restrict__ qp, int descending,
                                                           double m2pd, uint32_t kmax, float *__restrict__ dens,
                                                           uint32_t *__restrict__ heavy,
                                                           uint32_t *__restrict__ n_heavy)
{
  __shared__ FullShared<CAP, FULL> S;
  const int64_t L = v.L, T = (L + AHF_SLAB - 1) / AHF_SLAB;
  const int64_t nch = (L - 2 + zn - 1) / zn;
  int64_t b = blockIdx.x;
  if (b < AHF_XCDS * per_f) {
    const int64_t w = (b % AHF_XCDS) * per_f + b / AHF_XCDS;
    if (w >= 2 * T * T) return; /* the whole workgroup */
    gather_slab<CAP, FULL>(v, w % T, (w / T) % T, w / (T * T) == 0 ? 0 : L - 1, S, pmask, p0, qp, descending, m2pd, kmax,
                           dens, heavy, n_heavy);
  } else {
    b -= AHF_XCDS * per_f;
    const int64_t w = (b % AHF_XCDS) * per_m + b / AHF_XCDS;
    if (w >= T * T * nch) return; /* the whole workgroup */
    gather_march<CAP, FULL>(v, w % T, (w / T) % T, T, w / (T * T), zn, S, pmask, p0, qp, descending, m2pd, kmax, dens,
                            heavy, n_heavy);
  }
}

/* inclusive prefix sum over the 64 lanes of a wavefront by DPP row shifts
 * (within each row of 16) and row broadcasts of lanes 15 and 31 into the
 * rows above (the GFX9 scan; register-only) */
__device__ __forceinline__ int32_t wave_incl_scan_dpp(int32_t v)
{
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false); /* row_shr:1 */
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false); /* row_shr:2 */
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false); /* row_shr:4 */
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false); /* row_shr:8 */
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false); /* row_bcast:15 into rows 1, 3 */
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false); /* row_bcast:31 into rows 2, 3 */
  return v;
}

__device__ inline double readlane_d(double x, int l)
{
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(x), l);
  return __hiloint2double(hi, lo);
}

__device__ inline int64_t readlane_i64(int64_t x, int l)
{
  const int lo = __builtin_amdgcn_readlane((int)(uint32_t)(uint64_t)x, l);
  const int hi = __builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)x >> 32), l);
  return (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint64_t)(uint32_t)lo);
}

/*
 * AHF's d = (float)((double)d + c) over the contributions cv of lanes
 * [0, mm), in lane order, for the whole wavefront (d and mm uniform).
 * Inside one binade of d the steps are integer increments of d/ulp that
 * depend on c alone (ahf_fold_lane), so a run of them is one prefix sum over
 * the lanes; exact ties take the parity of the running value, lane by lane.
 * The first lane whose step leaves the binade (or whose start is zero or
 * subnormal) takes the plain FP32 step, and the fold resumes after it.
 * Every round settles at least one lane.  Lanes before `start` are settled.
 */
__device__ float fold_wave(float d, double cv, int start, int mm)
{
  const int lane = threadIdx.x & 63;
  while (start < mm) {
    int ok;
    const int e = ahf_fold_exponent(d, &ok);
    if (!ok) {
      d = (float)((double)d + readlane_d(cv, start));
      start++;
      continue;
    }
    const int neg = d < 0.0f;
    const int64_t K0 = ahf_fold_K(d, e);
    const bool act = lane >= start && lane < mm;
    int64_t R = 0, r = 0;
    int tie = 0, lok = 0;
    if (act) lok = ahf_fold_lane(cv, e, &R, &r, &tie);
    uint64_t tmask = __ballot(act && lok && tie);
    while (tmask) {
      const int l = __ffsll((unsigned long long)tmask) - 1;
      const uint64_t below = __ballot(act && (r & 1)) & ((1ull << l) - 1);
      const int par = (int)((K0 & 1) ^ (int64_t)(__popcll(below) & 1));
      const int64_t rl = readlane_i64(r, l);
      if (lane == l && ((par + (int)(rl & 1)) & 1)) r += 1;
      tmask &= tmask - 1;
    }
    /* a step that stays in the binade has |r| < 2^23, so r clamped to
     * +-2^24 keeps every prefix up to the first step that leaves it exact,
     * and 64 clamped steps fit in 32 bits */
    const int32_t rc = (int32_t)(r > ((int64_t)1 << 24) ? ((int64_t)1 << 24) : (r < -((int64_t)1 << 24) ? -((int64_t)1 << 24) : r));
    const int32_t Pi = wave_incl_scan_dpp(act ? rc : 0);
    const int64_t Kin = K0 + (int64_t)(Pi - (act ? rc : 0));
    const int valid = act && lok && ahf_fold_K_in(Kin, neg) && ahf_fold_T_in(Kin, R, neg);
    const uint64_t badm = __ballot(act && !valid);
    const int bad = badm ? __ffsll((unsigned long long)badm) - 1 : mm;
    if (bad > start) d = (float)ldexp((double)(K0 + (int64_t)__builtin_amdgcn_readlane(Pi, bad - 1)), e - 23);
    if (bad < mm) {
      d = (float)((double)d + readlane_d(cv, bad));
      start = bad + 1;
    } else {
      start = mm;
    }
  }
  return d;
}

/*
 * Heavy targets (more than kmax contributions), in two lists of one array:
 * those of at most AHF_HUGE contributions from its front, one wavefront
 * each, the larger ones from its back, one workgroup each.
 *
 * A target's contributions are flattened across its 27 sources in AHF's
 * visiting order (ahf_axis_order on each axis, z outer) and each source's
 * list order.  A wavefront takes AHF_HV * 64 of them at a time, contribution
 * base + 64*i + lane in register i.  As long as none is negative, none is an
 * exact tie and the value stays inside its binade, the block moves the
 * value's integer K by the sum of their steps (ahf_fold_step) in any order:
 * no scan over the lanes and no chain.  A block that fails the test is folded
 * 64 at a time in order (fold_wave): the first blocks, where the value runs
 * from -1 through zero, and then about one per doubling of the density.
 *
 * Bound by the latency of the folds and of the loads, so by the wavefronts in
 * flight: registers are held to 64 (8 wavefronts a SIMD; 81 registers and 5
 * wavefronts take 5.2 ms where this takes 4.2).  Measured over the levels of a
 * 192^3 clustered box (16,558 domain nodes above 384 contributions, the largest
 * 570,521): 24 ms with one wavefront and fold_wave for every 64 contributions
 * of a node, 4.2 ms now.
 */
#define AHF_HV 4
#define AHF_HBLK (64 * AHF_HV)
#define AHF_HEAVY_BS 512
#define AHF_HEAVY_NW (AHF_HEAVY_BS / 64)
/* a target's sources in LDS: exclusive prefix of the entry counts (off[27]
 * the total; an empty source shares its prefix with the next), the first
 * entry, the offset code of each, and the centres of the nodes at -1, 0, +1
 * along each axis */
struct HeavyTab {
  int64_t off[28], q0[27];
  double c[3][3]; /* x, y, z */
  int32_t code[27], pad;
};

/* by one wavefront; returns the total */
__device__ inline int64_t heavy_table(const level_view &v, const uint32_t *__restrict__ pmask,
                                      const int64_t *__restrict__ p0, int64_t n, int descending, HeavyTab *T)
{
  const int lane = threadIdx.x & 63;
  const int64_t o = n >> 3;
  const int c = (int)(n & 7);
  int64_t X, Y, Z;
  ahf_node_xyz(&v, o, c, &X, &Y, &Z);
  int64_t q0 = 0, cnt = 0;
  int code = 0;
  if (lane < 27) {
    int oz[3], oy[3], ox[3];
    ahf_axis_order(Z, v.L, oz);
    ahf_axis_order(Y, v.L, oy);
    ahf_axis_order(X, v.L, ox);
    const int ez = oz[lane / 9], ey = oy[(lane / 3) % 3], ex = ox[lane % 3];
    code = (ez + 1) * 16 + (ey + 1) * 4 + (ex + 1);
    const int64_t s = ahf_nbr_node(v.nbr, o, c, ex, ey, ez);
    if (s >= 0 && ((pmask[s] >> ((1 - ez) * 9 + (1 - ey) * 3 + (1 - ex))) & 1u)) {
      q0 = p0[s];
      cnt = p0[s + 1] - q0;
    }
  }
  int64_t inc = cnt;
#pragma unroll
  for (int d = 1; d < 32; d <<= 1) {
    const int64_t t = __shfl_up(inc, d, 64);
    if (lane >= d) inc += t;
  }
  const int64_t total = readlane_i64(inc, 26);
  if (lane < 27) {
    T->off[lane] = inc - cnt;
    T->q0[lane] = descending ? q0 + cnt - 1 : q0; /* the first in list order */
    T->code[lane] = code;
  } else if (lane == 27) {
    T->off[27] = total;
  } else if (lane >= 32 && lane < 41) {
    const int a = (lane - 32) / 3, k = (lane - 32) % 3;
    const int64_t W = a == 0 ? X : (a == 1 ? Y : Z);
    T->c[a][k] = ahf_centre(ahf_wrap(W - 1 + k, v.L), (double)v.L);
  }
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
  return total;
}

/* the contributions [base, base + AHF_HBLK) of a target, 0.0 past its last
 * (adding 0.0 leaves the value and K alone); j0: a source at or before the
 * one holding `base`, the same on every lane, moved up to it */
template <class Contrib>
__device__ __forceinline__ void heavy_fetch(const HeavyTab *T, int64_t total, int64_t base, int descending, int &j0,
                                            Contrib contrib, double cv[AHF_HV])
{
  const int lane = threadIdx.x & 63;
  while (j0 < 26 && T->off[j0 + 1] <= base) j0++;
  const bool one = T->off[j0 + 1] >= base + AHF_HBLK;
#pragma unroll
  for (int i = 0; i < AHF_HV; i++) {
    const int64_t k = base + 64 * i + lane;
    int j = j0;
    if (!one) {
      /* the last source whose prefix is at most k */
#pragma unroll
      for (int s = 16; s > 0; s >>= 1)
        if (j + s < 27 && T->off[j + s] <= k) j += s;
    }
    cv[i] = 0.0;
    if (k < total) {
      const int64_t kk = k - T->off[j];
      cv[i] = contrib(descending ? T->q0[j] - kk : T->q0[j] + kk, T->code[j]);
    }
  }
}

/* sum of the block's steps in the binade of exponent e over the wavefront;
 * 0 when some contribution rules the block sum out */
__device__ __forceinline__ int heavy_block_sum(const double cv[AHF_HV], int e, int64_t *S)
{
  const double scale = __longlong_as_double((long long)(1023 + 23 - e) << 52); /* 2^(23-e), -126 <= e <= 127 */
  int32_t s = 0;
  int ok = 1;
#pragma unroll
  for (int i = 0; i < AHF_HV; i++) {
    int32_t r;
    ok &= ahf_fold_step(cv[i], scale, &r) & (int)(cv[i] >= 0.0);
    s += r; /* at most 2^22 each */
  }
  /* at most 2^31 over the wavefront: exact modulo 2^32 */
  *S = (int64_t)(uint32_t)__builtin_amdgcn_readlane(wave_incl_scan_dpp(s), 63);
  return __ballot(!ok) == 0ull;
}

/* K of a normal float in its binade, and back */
__device__ __forceinline__ int64_t heavy_K(float d)
{
  const uint32_t u = __float_as_uint(d);
  const int64_t m = (int64_t)((u & 0x7FFFFFu) | 0x800000u);
  return (u >> 31) ? -m : m;
}
__device__ __forceinline__ float heavy_value(int64_t K, int e) { return ldexpf((float)(int32_t)K, e - 23); }

/*
 * 64 contributions in order (lanes [0, mm), the other lanes 0.0): rounds of a
 * scan of the steps over the lanes, each up to the first lane that ends on or
 * beyond the binade's edge, which takes the plain FP32 step; from a lane with
 * an exact tie (or a NaN) on by fold_wave, which knows the ties' parities.
 * A round is about 60 instructions; fold_wave's, on 64-bit integers, three
 * times that.
 */
__device__ __forceinline__ float heavy_fold1(float d, double cv, int mm)
{
  const int lane = threadIdx.x & 63;
  for (int start = 0; start < mm;) {
    int normal;
    const int e = ahf_fold_exponent(d, &normal);
    int bad = start;
    if (normal) {
      const double scale = __longlong_as_double((long long)(1023 + 23 - e) << 52);
      int32_t r;
      const int ok = ahf_fold_step(cv, scale, &r);
      const bool act = lane >= start;
      const int32_t P = wave_incl_scan_dpp(act ? r : 0); /* at most 2^28 */
      const int32_t K0 = (int32_t)heavy_K(d), K = K0 + P, A = K < 0 ? -K : K;
      /* strictly inside, of d's own sign: the double sum lay inside as well */
      const bool in = ok && A > (1 << 23) && A < (1 << 24) && (K ^ K0) >= 0;
      const uint64_t out = __ballot(act && lane < mm && !in);
      bad = out ? __builtin_ctzll(out) : mm;
      if (bad > start) d = heavy_value(K0 + (int64_t)__builtin_amdgcn_readlane(P, bad - 1), e);
      if (bad == mm) break;
      /* |c| of 2^22 ulps or more leaves the step to plain FP32 as well */
      const double c = readlane_d(cv, bad);
      if (!__builtin_amdgcn_readlane(ok, bad) && !(fabs(c * scale) >= 4194304.0)) return fold_wave(d, cv, bad, mm);
    }
    d = (float)((double)d + readlane_d(cv, bad));
    start = bad + 1;
  }
  return d;
}

/* the same one contribution after the other, the lanes read in turn: about 40
 * cycles each.  A target's first 64 run from -1 through zero and cross a
 * binade every few contributions; a round of heavy_fold1 for each crossing,
 * about 600 cycles, costs them four times as much. */
__device__ __forceinline__ float heavy_serial(float d, double cv, int mm)
{
  int l = 0;
  for (; l + 8 <= mm; l += 8)
#pragma unroll
    for (int i = 0; i < 8; i++) d = (float)((double)d + readlane_d(cv, l + i));
  for (; l < mm; l++) d = (float)((double)d + readlane_d(cv, l));
  return d;
}

/* the block folded 64 at a time, in order (cv is used up: rotated through
 * its first register, so the fold is there once and not AHF_HV times);
 * first: the target's first block */
__device__ __forceinline__ float heavy_fold64(float d, double cv[AHF_HV], int64_t left, bool first)
{
#pragma unroll 1
  for (int done = 0; done < AHF_HBLK && done < left; done += 64) {
    const int mm = (int)(left - done < 64 ? left - done : 64);
    d = first && done == 0 ? heavy_serial(d, cv[0], mm) : heavy_fold1(d, cv[0], mm);
#pragma unroll
    for (int i = 0; i + 1 < AHF_HV; i++) cv[i] = cv[i + 1];
  }
  return d;
}

template <class Contrib>
__device__ float heavy_wave(const HeavyTab *T, int64_t total, int descending, Contrib contrib)
{
  float d = -1.0f;
  int j0 = 0;
  for (int64_t base = 0; base < total; base += AHF_HBLK) {
    double cv[AHF_HV];
    heavy_fetch(T, total, base, descending, j0, contrib, cv);
    int ok;
    const int e = ahf_fold_exponent(d, &ok);
    if (ok) {
      int64_t S;
      ok = heavy_block_sum(cv, e, &S);
      const int64_t K = heavy_K(d);
      ok = ok && ahf_fold_block_in(K, S);
      if (ok) d = heavy_value(K + S, e);
    }
    if (!ok) d = heavy_fold64(d, cv, total - base, base == 0);
  }
  return d;
}

/* the same by the whole workgroup, its wavefronts taking consecutive blocks:
 * every wavefront sums its block in the binade the value has now, all of them
 * add the sums up in order to the first block that fails, that one is folded
 * by its wavefront, and the blocks after it are summed again in the binade
 * the value has then (at most AHF_HEAVY_NW rounds).  d and every branch
 * around a barrier are the same on all threads.  The rounds alternate
 * between two sets of words: a wavefront writes one of them only after the
 * barrier that follows every reading of the round before. */
struct HeavyRound {
  uint32_t S[2][AHF_HEAVY_NW];
  int32_t ok[2][AHF_HEAVY_NW];
  float d[2];
};

template <class Contrib>
__device__ float heavy_group(const HeavyTab *T, int64_t total, int descending, HeavyRound *R, int &turn,
                             Contrib contrib)
{
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  float d = -1.0f;
  int j0 = 0;
  for (int64_t base = 0; base < total; base += (int64_t)AHF_HEAVY_NW * AHF_HBLK) {
    double cv[AHF_HV];
    const int64_t wbase = base + (int64_t)w * AHF_HBLK;
    heavy_fetch(T, total, wbase, descending, j0, contrib, cv);
    for (int w0 = 0; w0 < AHF_HEAVY_NW; turn ^= 1) {
      int normal;
      const int e = ahf_fold_exponent(d, &normal);
      int64_t S = 0;
      int ok = 0;
      if (normal && w >= w0) ok = heavy_block_sum(cv, e, &S);
      if (lane == 0) {
        R->S[turn][w] = (uint32_t)S;
        R->ok[turn][w] = ok;
      }
      __syncthreads();
      int wb = w0;
      if (normal) {
        /* the value after each block from w0 on, one per lane (a sum of 2^24
         * or more, capped there, fails as it is); the first that fails */
        const bool mine = lane >= w0 && lane < AHF_HEAVY_NW;
        const uint32_t Sl = mine ? R->S[turn][lane] : 0u;
        const int okl = mine ? R->ok[turn][lane] : 0;
        const int32_t P = wave_incl_scan_dpp((int32_t)(Sl < (1u << 24) ? Sl : (1u << 24)));
        const int64_t K = heavy_K(d);
        const uint64_t fail = __ballot(mine && !(okl && ahf_fold_block_in(K, (int64_t)P)));
        wb = fail ? __builtin_ctzll(fail) : AHF_HEAVY_NW;
        if (wb > w0) d = heavy_value(K + (int64_t)__builtin_amdgcn_readlane(P, wb - 1), e);
      }
      if (wb < AHF_HEAVY_NW) {
        if (w == wb) {
          const float f = heavy_fold64(d, cv, total - wbase, wbase == 0);
          if (lane == 0) R->d[turn] = f;
        }
        __syncthreads();
        d = R->d[turn];
      }
      w0 = wb + 1;
    }
  }
  return d;
}

/*
 * Exact-order density of the heavy targets: first the huge ones by
 * workgroups, then the others by wavefronts.  Every level's heavy targets
 * read the 16-byte position records, consecutive lanes consecutive records,
 * and form the weights again (about 40 FP64 instructions): over 80-byte
 * weight records a wavefront's loads touch five times the cache lines.
 */
__global__ void __launch_bounds__(AHF_HEAVY_BS, 8) k_gather_heavy(level_view v, const uint32_t *__restrict__ pmask,
                                                               const int64_t *__restrict__ p0,
                                                               const ahf_q4 *__restrict__ qp, int descending,
                                                               double m2pd, float *__restrict__ dens,
                                                               const uint32_t *__restrict__ heavy,
                                                               const uint32_t *__restrict__ n_heavy)
{
  __shared__ HeavyTab s_tab[AHF_HEAVY_NW];
  __shared__ HeavyRound s_round;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  HeavyTab *T = s_tab + w;
  const int64_t n_huge = (int64_t)n_heavy[1], n_rest = (int64_t)n_heavy[0], nn = 8 * v.n_oct;
  const double L = (double)v.L;
  auto contrib = [=](int64_t q, int code) {
    const ahf_q4 r = qp[q];
    const int ez = (code >> 4) - 1, ey = ((code >> 2) & 3) - 1, ex = (code & 3) - 1;
    const double wz = TscRt(-ez)(ahf_pn_sep(r.z, T->c[2][ez + 1], L));
    const double wy = TscRt(-ey)(ahf_pn_sep(r.y, T->c[1][ey + 1], L));
    const double wx = TscRt(-ex)(ahf_pn_sep(r.x, T->c[0][ex + 1], L));
    return ((m2pd * wz) * wy) * wx;
  };
  int turn = 0;
  for (int64_t i = blockIdx.x; i < n_huge; i += gridDim.x) {
    const int64_t n = heavy[nn - 1 - i];
    const int64_t total = heavy_table(v, pmask, p0, n, descending, T);
    const float d = heavy_group(T, total, descending, &s_round, turn, contrib);
    if (threadIdx.x == 0) dens[n] = d;
  }
  for (int64_t i = (int64_t)w * gridDim.x + blockIdx.x; i < n_rest; i += (int64_t)gridDim.x * AHF_HEAVY_NW) {
    const int64_t n = heavy[i];
    const int64_t total = heavy_table(v, pmask, p0, n, descending, T);
    const float d = heavy_wave(T, total, descending, contrib);
    if (lane == 0) dens[n] = d;
  }
}

/*
 * ahf_node_flags for the 8 children of one octet per thread: a child with
 * all 27 neighbours present is interior, and tested when one of its 18
 * neighbours at x offsets 0, +1 reaches the density threshold.  The
 * children's neighbours lie in the 3x4x4 nodes from (X0, Y0-1, Z0) (X0,
 * Y0, Z0 the octet's first node), each density read once.  Missing
 * neighbour octets only occur for children that are not interior.
 */
__global__ void k_flags(level_view v, const uint32_t *__restrict__ pmask, const float *__restrict__ dens,
                        double thr, uint8_t *__restrict__ flags)
{
  const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (o >= v.n_oct) return;
  const uint4 *pm4 = reinterpret_cast<const uint4 *>(pmask + 8 * o);
  const uint4 pa = pm4[0], pb = pm4[1];
  const uint32_t pm[8] = {pa.x, pa.y, pa.z, pa.w, pb.x, pb.y, pb.z, pb.w};
  uint32_t any = 0;
#pragma unroll
  for (int c = 0; c < 8; c++) any |= (pm[c] == AHF_FULL27) ? 1u << c : 0u;
  uint64_t hit = 0; /* bit xi + 3*(yi + 4*zi) of the 3x4x4 neighbourhood */
  if (any) {
    int32_t nb[27];
#pragma unroll
    for (int i = 0; i < 27; i++) nb[i] = v.nbr[27 * o + i];
    /* every load issued at once: a missing octet reads this octet's node
     * and its bit is dropped */
    float dv[48];
#pragma unroll
    for (int zi = 0; zi < 4; zi++)
#pragma unroll
      for (int yi = 0; yi < 4; yi++)
#pragma unroll
        for (int xi = 0; xi < 3; xi++) {
          const int zr = zi - 1, yr = yi - 1, xr = xi;
          const int oz = zr < 0 ? -1 : (zr > 1 ? 1 : 0), oy = yr < 0 ? -1 : (yr > 1 ? 1 : 0), oxo = xr > 1 ? 1 : 0;
          const int32_t on = nb[ahf_e27(oxo, oy, oz)];
          const int64_t m = 8 * (int64_t)(on >= 0 ? on : (int32_t)o) + ((zr & 1) << 2 | (yr & 1) << 1 | (xr & 1));
          dv[xi + 3 * (yi + 4 * zi)] = dens[m];
        }
#pragma unroll
    for (int zi = 0; zi < 4; zi++)
#pragma unroll
      for (int yi = 0; yi < 4; yi++)
#pragma unroll
        for (int xi = 0; xi < 3; xi++) {
          const int zr = zi - 1, yr = yi - 1, xr = xi;
          const int oz = zr < 0 ? -1 : (zr > 1 ? 1 : 0), oy = yr < 0 ? -1 : (yr > 1 ? 1 : 0), oxo = xr > 1 ? 1 : 0;
          const int bit = xi + 3 * (yi + 4 * zi);
          if (nb[ahf_e27(oxo, oy, oz)] >= 0 && (double)dv[bit] >= thr) hit |= 1ull << bit;
        }
  }
  uint8_t f[8];
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const int cx = c & 1, cy = (c >> 1) & 1, cz = c >> 2;
    /* xi in {cx, cx+1}, yi in {cy..cy+2}, zi in {cz..cz+2} */
    uint64_t box = 0;
#pragma unroll
    for (int zi = 0; zi < 3; zi++)
#pragma unroll
      for (int yi = 0; yi < 3; yi++) box |= 3ull << (cx + 3 * (cy + yi + 4 * (cz + zi)));
    f[c] = !((any >> c) & 1u) ? (uint8_t)0 : (uint8_t)(NF_INTERIOR | ((hit & box) ? NF_TEST : 0u));
  }
  uint2 w;
  w.x = (uint32_t)f[0] | (uint32_t)f[1] << 8 | (uint32_t)f[2] << 16 | (uint32_t)f[3] << 24;
  w.y = (uint32_t)f[4] | (uint32_t)f[5] << 8 | (uint32_t)f[6] << 16 | (uint32_t)f[7] << 24;
  *reinterpret_cast<uint2 *>(flags + 8 * o) = w;
}

/* one thread per level row (octet row r, cy, cz) */
__global__ void k_refine_rows(level_view v, uint8_t *__restrict__ flags, int64_t *__restrict__ cnt,
                              int32_t *__restrict__ anomaly)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 4 * v.n_row) return;
  const int64_t r = t >> 2;
  const int cy = (int)(t & 1), cz = (int)((t >> 1) & 1);
  int64_t c = 0;
  if (ahf_plane_tested(&v, v.row_plane[r], cz) && ahf_row_tested(&v, r, cy)) {
    int an = 0;
    c = ahf_refine_row(&v, flags, r, cy, cz, &an);
    if (an) atomicOr(anomaly, 1);
  }
  cnt[ahf_row_rank(&v, r, cy, cz)] = c;
}

/* has-flag of every level plane (octet plane p, cz) */
__global__ void k_plane_has(level_view v, const int64_t *__restrict__ cnt, int32_t *__restrict__ has)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 2 * v.n_plane) return;
  const int64_t p = t >> 1;
  const int cz = (int)(t & 1);
  const int64_t q0 = v.plane_row0[p], nr = v.plane_row0[p + 1] - q0;
  const int64_t r0 = 4 * q0 + cz * 2 * nr;
  int32_t h = 0;
  for (int64_t k = 0; k < 2 * nr && !h; k++) h = cnt[r0 + k] > 0;
  has[t] = h;
}

__global__ void k_nonzero(const int64_t *__restrict__ cnt, int64_t n, int32_t *__restrict__ out)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = cnt[i] > 0;
}

/* writes the next level's octets, octet rows and node2oct of this level */
__global__ void k_compact(level_view v, const uint8_t *__restrict__ flags, const int64_t *__restrict__ cnt,
                          const int64_t *__restrict__ oct_off, const int32_t *__restrict__ row_off,
                          const int32_t *__restrict__ plane_off, uint64_t *__restrict__ key2,
                          uint8_t *__restrict__ link2, int64_t *__restrict__ parent2, uint64_t *__restrict__ rkey2,
                          int32_t *__restrict__ roct2, int32_t *__restrict__ rplane2, int32_t *__restrict__ node2oct)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 4 * v.n_row) return;
  const int64_t r = t >> 2;
  const int cy = (int)(t & 1), cz = (int)((t >> 1) & 1);
  const int64_t rank = ahf_row_rank(&v, r, cy, cz);
  if (cnt[rank] == 0) return;
  const int64_t p = v.row_plane[r];
  const int64_t Y = 2 * ahf_row_y(v.row_key[r]) + cy, Z = 2 * (int64_t)v.plane_z[p] + cz;
  const int64_t nr = row_off[rank];
  int64_t w = oct_off[rank];
  rkey2[nr] = (uint64_t)Y | ((uint64_t)Z << AHF_KEY_BITS);
  roct2[nr] = (int32_t)w;
  rplane2[nr] = plane_off[2 * p + cz];
  for (int64_t o = v.row_oct0[r]; o < v.row_oct0[r + 1]; o++)
    for (int cx = 0; cx < 2; cx++) {
      const int64_t nd = 8 * o + cz * 4 + cy * 2 + cx;
      const uint8_t f = flags[nd];
      if (!(f & NF_REFINED)) continue;
      const int64_t X = 2 * ahf_kx(v.oct_key[o]) + cx;
      key2[w] = ahf_pack3((uint64_t)X, (uint64_t)Y, (uint64_t)Z);
      link2[w] = (f & NF_LINK) ? 1 : 0;
      parent2[w] = nd;
      node2oct[nd] = (int32_t)w;
      w++;
    }
}

__global__ void k_plane_fill(level_view v, const int32_t *__restrict__ has, const int32_t *__restrict__ plane_off,
                             const int32_t *__restrict__ row_off, int32_t *__restrict__ pz2,
                             int32_t *__restrict__ prow2)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 2 * v.n_plane || !has[t]) return;
  const int64_t p = t >> 1;
  const int cz = (int)(t & 1);
  const int64_t q0 = v.plane_row0[p], nr = v.plane_row0[p + 1] - q0;
  const int32_t np = plane_off[t];
  pz2[np] = 2 * v.plane_z[p] + cz;
  prow2[np] = row_off[4 * q0 + cz * 2 * nr];
}

/* the refine step's sizes gathered for one read-back */
__global__ void k_sizes(const int64_t *__restrict__ n_oct, const int64_t *__restrict__ n_part,
                        const int32_t *__restrict__ n_row, const int32_t *__restrict__ n_plane,
                        const int32_t *__restrict__ anomaly, int64_t *__restrict__ out)
{
  out[0] = *n_oct;
  out[1] = *n_part;
  out[2] = *n_row;
  out[3] = *n_plane;
  out[4] = *anomaly;
}

__global__ void k_set2(int32_t *__restrict__ a, int64_t ia, int32_t va, int32_t *__restrict__ b, int64_t ib,
                       int32_t vb)
{
  a[ia] = va;
  b[ib] = vb;
}

__global__ void k_nbr_next(const int32_t *__restrict__ nbr, const int64_t *__restrict__ parent2,
                           const int32_t *__restrict__ node2oct, int64_t n2, int32_t *__restrict__ nbr2)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 27 * n2) return;
  const int64_t o2 = t < (int64_t)UINT32_MAX ? (int64_t)((uint32_t)t / 27u) : t / 27;
  const int e = (int)(t - 27 * o2);
  const int ex = e % 3 - 1, ey = (e / 3) % 3 - 1, ez = e / 9 - 1;
  const int64_t pn = parent2[o2];
  const int64_t m = ahf_nbr_node(nbr, pn >> 3, (int)(pn & 7), ex, ey, ez);
  nbr2[t] = m < 0 ? -1 : node2oct[m];
}

/* relink (src/libamr_serial/relink.c:31-288): per bucket entry, the fine
 * child its particle moves to (first interior child, in fine traversal
 * order, whose closed cell holds it); the key for the stable sort that
 * builds the fine buckets is the fine node, or all-ones if it stays */
/* imask2: interior children of each fine octet (k_pmask); qp: the
 * entries' position records when the level has them, else the particle
 * arrays are read */
__global__ void k_relink_child(int64_t n_ent, const uint32_t *__restrict__ pnode,
                               const uint32_t *__restrict__ plist, const int32_t *__restrict__ node2oct,
                               const uint64_t *__restrict__ key, const uint8_t *__restrict__ imask2,
                               const ahf_q4 *__restrict__ qp, const float *__restrict__ px,
                               const float *__restrict__ py, const float *__restrict__ pz, double Lf,
                               int8_t *__restrict__ child)
{
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n_ent) return;
  const uint32_t m = pnode[q];
  const int32_t o2 = node2oct[m];
  int ch = -1;
  if (o2 >= 0) {
    const uint8_t imask = imask2[o2];
    if (imask) {
      const uint64_t mk = key[m >> 3];
      const int cm = (int)(m & 7);
      const int64_t MX = 2 * ahf_kx(mk) + (cm & 1), MY = 2 * ahf_ky(mk) + ((cm >> 1) & 1),
                    MZ = 2 * ahf_kz(mk) + (cm >> 2);
      float x, y, z;
      if (qp) {
        const ahf_q4 r = qp[q];
        x = r.x;
        y = r.y;
        z = r.z;
      } else {
        const uint32_t p = plist[q];
        x = px[p];
        y = py[p];
        z = pz[p];
      }
      ch = ahf_relink_child_h(x, y, z, MX, MY, MZ, Lf, imask);
    }
  }
  child[q] = (int8_t)ch;
}

/*
 * Fine buckets without a sort: a particle only moves to a child of its own
 * node, so fine node t = 8*o2 + c holds the entries of its mother's bucket
 * whose child is c, in bucket order (AHF's head insertion during relink
 * leaves them in this order relative to the walk).  One thread per fine
 * octet walks the mother's bucket once to count its 8 children; after a scan,
 * each entry finds its place from the earlier entries of its bucket.  Buckets of more
 * than AHF_BIG_BUCKET entries are listed for k_fine_big, which walks them
 * one wavefront at a time, and those of more than AHF_HUGE_BUCKET, listed from
 * the other end, one workgroup at a time.
 */
#define AHF_BIG_BUCKET 32
#define AHF_HUGE_BUCKET 1024
#define AHF_FINE_BS 512
#define AHF_FINE_BLOCKS 512 /* for either list */

__global__ void k_fine_count(const int64_t *__restrict__ oct_parent, int64_t n2, const int64_t *__restrict__ p0c,
                             const int8_t *__restrict__ child, int64_t *__restrict__ cnt,
                             uint32_t *__restrict__ big, uint32_t *__restrict__ n_big)
{
  const int64_t t8 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t8 >= n2) return;
  const int64_t m = oct_parent[t8];
  const int64_t a = p0c[m], b = p0c[m + 1];
  if (b - a > AHF_BIG_BUCKET) {
    if (b - a > AHF_HUGE_BUCKET) big[n2 - 1 - (int64_t)atomicAdd(n_big + 1, 1u)] = (uint32_t)t8;
    else big[atomicAdd(n_big, 1u)] = (uint32_t)t8;
    return;
  }
  /* the 8 children's counts as 16-bit fields (at most AHF_BIG_BUCKET) */
  uint64_t lo = 0, hi = 0;
  for (int64_t q = a; q < b; q++) {
    const int c = child[q];
    if (c < 0) continue;
    if (c < 4) lo += 1ull << (16 * c);
    else hi += 1ull << (16 * (c - 4));
  }
#pragma unroll
  for (int c = 0; c < 4; c++) {
    cnt[8 * t8 + c] = (int64_t)((lo >> (16 * c)) & 0xFFFFu);
    cnt[8 * t8 + 4 + c] = (int64_t)((hi >> (16 * c)) & 0xFFFFu);
  }
}

/* one thread per coarse bucket entry: its place in the fine bucket of its
 * child is the fine bucket's start plus the number of earlier entries of
 * the mother's bucket with the same child (buckets over AHF_BIG_BUCKET
 * entries are k_fine_big's) */
__global__ void k_fine_fill(int64_t n_ent, const uint32_t *__restrict__ pnode, const int32_t *__restrict__ node2oct,
                            const int64_t *__restrict__ p0c, const int8_t *__restrict__ child,
                            const uint32_t *__restrict__ plistc, const int64_t *__restrict__ p0f,
                            uint32_t *__restrict__ plistf, uint32_t *__restrict__ pnodef)
{
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n_ent) return;
  const int c = child[q];
  if (c < 0) return;
  const uint32_t m = pnode[q];
  const int64_t a = p0c[m];
  if (p0c[m + 1] - a > AHF_BIG_BUCKET) return;
  const int64_t t = 8 * (int64_t)node2oct[m] + c;
  int64_t rank = 0;
  for (int64_t k = a; k < q; k++) rank += child[k] == c;
  const int64_t w = p0f[t] + rank;
  plistf[w] = plistc[q];
  pnodef[w] = (uint32_t)t;
}

/*
 * One bucket by a workgroup: 8 consecutive entries a thread, the children's
 * counts as 16-bit fields of two words (at most 4096 each), the next step's
 * child numbers loaded before this step's are ranked.  The counts need no
 * barrier before the end; the places take one scan over the workgroup a step.
 * A serial chain over the bucket: one wavefront's steps of 64 entries took
 * 3.6 ms of a clustered 192^3 box's build (buckets of up to some 10^5
 * entries).
 */
struct FinePack {
  uint64_t lo, hi;
};

__device__ __forceinline__ FinePack fine_pack(const int8_t ch[8])
{
  FinePack p = {0, 0};
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int c = ch[i];
    const uint64_t one = c >= 0 ? 1ull << (16 * (c & 3)) : 0ull;
    if (c < 4) p.lo += one;
    else p.hi += one;
  }
  return p;
}

__device__ __forceinline__ int64_t fine_field(const FinePack &p, int c)
{
  return (int64_t)(((c < 4 ? p.lo : p.hi) >> (16 * (c & 3))) & 0xFFFFu);
}

__device__ __forceinline__ void fine_load(const int8_t *__restrict__ child, int64_t q, int64_t b, int8_t ch[8])
{
#pragma unroll
  for (int i = 0; i < 8; i++) ch[i] = q + i < b ? child[q + i] : (int8_t)-1;
}

template <bool FILL>
__device__ __forceinline__ void fine_group(int64_t o2, int64_t a, int64_t b, const int8_t *__restrict__ child,
                                           const uint32_t *__restrict__ plistc, int64_t *__restrict__ cnt,
                                           const int64_t *__restrict__ p0f, uint32_t *__restrict__ plistf,
                                           uint32_t *__restrict__ pnodef)
{
  constexpr int NW = AHF_FINE_BS / 64, STEP = AHF_FINE_BS * 8;
  __shared__ FinePack s_tot[2][NW];
  __shared__ unsigned long long s_cnt[8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if constexpr (!FILL) {
    if (threadIdx.x < 8) s_cnt[threadIdx.x] = 0;
    uint32_t c8[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t q = a + 8 * (int64_t)threadIdx.x; q < b; q += STEP) {
      int8_t ch[8];
      fine_load(child, q, b, ch);
      const FinePack p = fine_pack(ch);
#pragma unroll
      for (int c = 0; c < 8; c++) c8[c] += (uint32_t)fine_field(p, c);
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 8; c++)
      if (c8[c]) atomicAdd(&s_cnt[c], (unsigned long long)c8[c]);
    __syncthreads();
    if (threadIdx.x < 8) cnt[8 * o2 + threadIdx.x] = (int64_t)s_cnt[threadIdx.x];
    __syncthreads();
  } else {
    int64_t run[8];
#pragma unroll
    for (int c = 0; c < 8; c++) run[c] = p0f[8 * o2 + c];
    int8_t nx[8];
    fine_load(child, a + 8 * (int64_t)threadIdx.x, b, nx);
    int buf = 0;
    for (int64_t q0 = a; q0 < b; q0 += STEP, buf ^= 1) {
      const int64_t q = q0 + 8 * (int64_t)threadIdx.x;
      int8_t ch[8];
#pragma unroll
      for (int i = 0; i < 8; i++) ch[i] = nx[i];
      uint32_t pl[8];
#pragma unroll
      for (int i = 0; i < 8; i++) pl[i] = ch[i] >= 0 ? plistc[q + i] : 0u;
      fine_load(child, q + STEP, b, nx);
      FinePack in = fine_pack(ch);
      const FinePack mine = in;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const uint64_t l = __shfl_up(in.lo, d, 64), h = __shfl_up(in.hi, d, 64);
        if (lane >= d) {
          in.lo += l;
          in.hi += h;
        }
      }
      if (lane == 63) s_tot[buf][wave] = in;
      __syncthreads();
      FinePack below = {in.lo - mine.lo, in.hi - mine.hi}, all = {0, 0};
#pragma unroll
      for (int w = 0; w < NW; w++) {
        const FinePack t = s_tot[buf][w];
        if (w < wave) {
          below.lo += t.lo;
          below.hi += t.hi;
        }
        all.lo += t.lo;
        all.hi += t.hi;
      }
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int c = ch[i];
        if (c < 0) continue;
        int64_t pos = fine_field(below, c);
#pragma unroll
        for (int k = 0; k < 8; k++) pos += k == c ? run[k] : 0;
        plistf[pos] = pl[i];
        pnodef[pos] = (uint32_t)(8 * o2 + c);
        if (c < 4) below.lo += 1ull << (16 * c);
        else below.hi += 1ull << (16 * (c - 4));
      }
#pragma unroll
      for (int c = 0; c < 8; c++) run[c] += fine_field(all, c);
    }
    __syncthreads(); /* the words are the next bucket's */
  }
}

/* the listed buckets: the first half of the workgroups a wavefront per big
 * bucket, 64 entries per step, each ranked among the earlier entries of its
 * child by ballots; the second half a workgroup per huge one.  FILL = false
 * writes the 8 counts, FILL = true the entries. */
template <bool FILL>
__global__ void __launch_bounds__(AHF_FINE_BS) k_fine_big(int64_t n2, const int64_t *__restrict__ oct_parent,
                                                        const int64_t *__restrict__ p0c,
                                                        const int8_t *__restrict__ child,
                                                        const uint32_t *__restrict__ plistc,
                                                        const uint32_t *__restrict__ big,
                                                        const uint32_t *__restrict__ n_big,
                                                        int64_t *__restrict__ cnt, const int64_t *__restrict__ p0f,
                                                        uint32_t *__restrict__ plistf,
                                                        uint32_t *__restrict__ pnodef)
{
  const int lane = threadIdx.x & 63;
  const uint64_t lt = (lane == 0) ? 0ull : ((~0ull) >> (64 - lane));
  const int64_t gw = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t nw = ((int64_t)AHF_FINE_BLOCKS * blockDim.x) >> 6;
  if (blockIdx.x >= AHF_FINE_BLOCKS) {
    const int64_t nh = (int64_t)n_big[1];
    for (int64_t i = blockIdx.x - AHF_FINE_BLOCKS; i < nh; i += AHF_FINE_BLOCKS) {
      const int64_t o2 = big[n2 - 1 - i], m = oct_parent[o2];
      fine_group<FILL>(o2, p0c[m], p0c[m + 1], child, plistc, cnt, p0f, plistf, pnodef);
    }
    return;
  }
  const int64_t nb = (int64_t)*n_big;
  for (int64_t i = gw; i < nb; i += nw) {
    const int64_t o2 = big[i];
    const int64_t m = oct_parent[o2];
    const int64_t a = p0c[m], b = p0c[m + 1];
    /* lane c < 8 keeps the running count of child c */
    int64_t run = 0, base = 0;
    if (FILL && lane < 8) base = p0f[8 * o2 + lane];
    for (int64_t q0 = a; q0 < b; q0 += 64) {
      const int64_t q = q0 + lane;
      const int ch = q < b ? (int)child[q] : -1;
      uint64_t bal[8];
#pragma unroll
      for (int k = 0; k < 8; k++) bal[k] = __ballot(ch == k);
      /* every lane takes part in the shuffle: the first free slot of its child */
      const int64_t slot = __shfl(base + run, ch >= 0 ? ch : 0, 64);
      if (FILL && ch >= 0) {
        uint64_t mine = bal[0];
#pragma unroll
        for (int k = 1; k < 8; k++) mine = ch == k ? bal[k] : mine;
        const int64_t pos = slot + (int64_t)__popcll(mine & lt);
        plistf[pos] = plistc[q];
        pnodef[pos] = (uint32_t)(8 * o2 + ch);
      }
      uint64_t my = bal[0];
#pragma unroll
      for (int k = 1; k < 8; k++) my = lane == k ? bal[k] : my;
      if (lane < 8) run += (int64_t)__popcll(my);
    }
    if (!FILL && lane < 8) cnt[8 * o2 + lane] = run;
  }
}

/* neighbour table of a standalone level: binary search of the periodic
 * neighbour key in the sorted octet keys */
__global__ void k_nbr_search(const uint64_t *__restrict__ key, int64_t n_oct, int64_t half,
                             int32_t *__restrict__ nbr)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 27 * n_oct) return;
  const int64_t o = t / 27;
  const int e = (int)(t % 27);
  const int ex = e % 3 - 1, ey = (e / 3) % 3 - 1, ez = e / 9 - 1;
  const uint64_t k = key[o];
  const uint64_t want = ahf_pack3((uint64_t)ahf_wrap(ahf_kx(k) + ex, half), (uint64_t)ahf_wrap(ahf_ky(k) + ey, half),
                                  (uint64_t)ahf_wrap(ahf_kz(k) + ez, half));
  int64_t lo = 0, hi = n_oct - 1, found = -1;
  while (lo <= hi) {
    const int64_t mid = (lo + hi) >> 1;
    const uint64_t km = key[mid];
    if (km == want) { found = mid; break; }
    if (km < want) lo = mid + 1; else hi = mid - 1;
  }
  nbr[t] = (int32_t)found;
}

/* ============================================================ host side */

static inline unsigned nblk(int64_t n)
{
  return (unsigned)((n + AHF_BLOCK - 1) / AHF_BLOCK);
}

#define LAUNCH(kern, n, ...)                                                                 \
  do {                                                                                       \
    if ((n) > 0) hipLaunchKernelGGL(kern, dim3(nblk(n)), dim3(AHF_BLOCK), 0, c->st, __VA_ARGS__); \
  } while (0)

static level_view make_view(const DevLevel &l)
{
  level_view v;
  v.L = l.L;
  v.n_oct = l.n_oct;
  v.oct_key = l.oct_key;
  v.oct_link = l.oct_link;
  v.nbr = l.nbr;
  v.n_row = l.n_row;
  v.row_key = l.row_key;
  v.row_oct0 = l.row_oct0;
  v.row_plane = l.row_plane;
  v.n_plane = l.n_plane;
  v.plane_z = l.plane_z;
  v.plane_row0 = l.plane_row0;
  return v;
}

/* bucket entries per node from which a level counts as dense */
#define AHF_DENSE_ENTRIES_PER_NODE 3
/* heavy-node workgroups: four of 8 wavefronts on each of 256 CUs, all resident */
#define AHF_HEAVY_BLOCKS 1024
/* nodes with more contributions than this go to the heavy kernel: on levels
 * that do not march, and at most on any */
#define AHF_KMAX_SMALL 96
#define AHF_KMAX_TOP 2000

/* a level that holds every octet takes the staged plane walk, unless it is
 * so small that its few workgroups, each marching through planes, take longer
 * than a lane or a wavefront per node */
/* L = 32 at 8 and at 1 entries a node: 0.54 ms marched, 0.09 ms not; L = 50:
 * 0.58 ms marched (deposit of all its levels), 0.96 ms not */
#define AHF_MARCH_MIN_L 40
static bool marches(const ahfgpu_ctx *c, int64_t L, int64_t n_oct)
{
  return c->gather_mode == AHFGPU_GATHER_AUTO && L >= AHF_MARCH_MIN_L && n_oct == (L / 2) * (L / 2) * (L / 2);
}

/* target planes per marching workgroup: a workgroup walks zn + 2 source
 * planes, and about AHF_MARCH_FILL of them are resident at once, so on small
 * levels the fewest rounds of planes (L = 64: 496 workgroups of 2 planes take
 * 0.15 ms, 128 of 8 planes 0.37).  Larger levels have workgroups to spare and
 * take the planes that re-read least. */
#define AHF_MARCH_FILL 512
static int64_t march_planes(int64_t L, int64_t side)
{
  if (L >= 128) return L <= 128 ? 8 : 16;
  int64_t best = 0, cost = 0;
  for (int64_t zn = 1; zn <= 16; zn *= 2) {
    const int64_t wg = side * side * ((L - 2 + zn - 1) / zn);
    const int64_t c = (wg + AHF_MARCH_FILL - 1) / AHF_MARCH_FILL * (zn + 2);
    if (!best || c < cost) {
      best = zn;
      cost = c;
    }
  }
  return best;
}

/*
 * Exact-order gather of one level over its n_ent bucket entries, a position
 * record each: levels that hold every octet and are not small march
 * (k_gather_full); on the others the octets are sorted into Morton order (the
 * target order), and then either
 *  - dense levels (many entries per node): the per-source walk
 *    (k_gather_src), whose records stay in L2; or
 *  - sparse levels: a TSC weight record per entry as well and the flat walk
 *    (k_gather_light), which keeps a wavefront's lanes busy when buckets
 *    hold a particle or two;
 * and by wavefronts the nodes with more than kmax contributions.  Every
 * choice gives the same bits.  Needs pmask.
 */
static int gather_level(ahfgpu_ctx *c, DevLevel &l, int64_t n_ent, int descending, bool timed)
{
  const int64_t nn = 8 * l.n_oct, no = l.n_oct;
  level_view v = make_view(l);
  Arena &A = c->arena;
  /* a level that holds every octet takes the staged plane walk */
  const bool slab = marches(c, l.L, no);
  const bool dense = slab || c->gather_mode == AHFGPU_GATHER_SOURCE ||
                     ((c->gather_mode == AHFGPU_GATHER_AUTO || c->gather_mode == AHFGPU_GATHER_WAVE) &&
                      n_ent >= AHF_DENSE_ENTRIES_PER_NODE * nn);
  l.dens = A.get<float>(nn);
  l.qp = A.get<ahf_q4>(n_ent > 0 ? n_ent : 1);
  l.W = dense ? nullptr : A.get<ahf_w9>(n_ent > 0 ? n_ent : 1);
  uint32_t *heavy = A.get<uint32_t>(nn);
  if (!l.dens || !l.qp || (!dense && !l.W) || !heavy) return AHFGPU_ENOMEM;
  uint32_t *n_heavy = (uint32_t *)(c->d_anomaly + 4); /* two counts */
  hipMemsetAsync(n_heavy, 0, 2 * sizeof(uint32_t), c->st);
  hipEvent_t e0 = timed ? c->timer_begin() : nullptr;
  if (dense)
    LAUNCH(k_prep_q, n_ent, l.node_p0 + nn, n_ent, l.plist, c->px, c->py, c->pz, l.qp);
  else
    LAUNCH(k_prep, n_ent, v, l.node_p0 + nn, n_ent, l.pnode, l.plist, c->px, c->py, c->pz, l.m2pd, l.W, l.qp);
  if (!l.tord) {
    /* no order inherited from a coarser level: sort the octets' Morton keys */
    uint64_t *mk0 = A.get<uint64_t>(no), *mk1 = A.get<uint64_t>(no);
    uint32_t *ix0 = A.get<uint32_t>(no), *ix1 = A.get<uint32_t>(no);
    uint32_t *rtmp = A.get<uint32_t>(radix_tmp_u32<uint64_t>(no));
    if (!mk0 || !mk1 || !ix0 || !ix1 || !rtmp) return AHFGPU_ENOMEM;
    int axis_bits = 1;
    while ((1ll << axis_bits) < l.L / 2) axis_bits++;
    LAUNCH(k_morton_keys, no, v, mk0, ix0);
    const int w = radix_sort<uint64_t, uint32_t>(mk0, ix0, mk1, ix1, no, 3 * axis_bits, rtmp, c->st);
    l.tord = w ? ix1 : ix0;
  }
  const uint32_t *tord = l.tord;
  if (timed)
    c->timer_end(e0, TIMER_PREP, (12.0 + 8.0 + (dense ? 16.0 : 80.0)) * (double)n_ent + 24.0 * (double)no);
  hipEvent_t e1 = timed ? c->timer_begin() : nullptr;
  const int64_t per_xcd = (nblk(nn) + AHF_XCDS - 1) / AHF_XCDS;
  const dim3 grid((unsigned)(AHF_XCDS * per_xcd));
  /* a lane's chain holds its whole wavefront, so a node goes to the heavy
   * kernel once it has well more contributions than its neighbours: half as
   * much again as the marching level's mean of 27 per entry of a node, and
   * AHF_KMAX_SMALL on the others (the schedule's kmax_big and kmax_small set the
   * threshold itself, for levels of 2^21 nodes or more and for smaller ones) */
  const int64_t mean = 27 * n_ent / (nn > 0 ? nn : 1);
  const uint32_t kdef =
      slab ? (uint32_t)std::min<int64_t>(AHF_KMAX_TOP, std::max<int64_t>(AHF_KMAX_SMALL, mean + mean / 2)) : AHF_KMAX_SMALL;
  const int32_t kset = nn >= ((int64_t)1 << 21) ? c->kmax_big : c->kmax_small;
  const uint32_t kmax = c->gather_mode == AHFGPU_GATHER_WAVE ? 0u : kset > 0 ? (uint32_t)kset : kdef;
  static_assert(AHF_KMAX_TOP < 4096, "the march's queue words hold counts below 4096");
  if (slab) {
    /* the planes 1..L-2 march, the two face planes take the per-plane walk */
    const int64_t side = (l.L + AHF_SLAB - 1) / AHF_SLAB;
    const int64_t zn = c->march_zn > 0 ? c->march_zn : march_planes(l.L, side), nch = (l.L - 2 + zn - 1) / zn;
    const int64_t per_m = (side * side * nch + AHF_XCDS - 1) / AHF_XCDS;
    const int64_t per_f = (side * side * 2 + AHF_XCDS - 1) / AHF_XCDS;
    const dim3 fgrid((unsigned)(AHF_XCDS * (per_f + per_m)));
    if (n_ent >= 2 * nn)
      hipLaunchKernelGGL((k_gather_full<AHF_FULL_CAP_BIG, false>), fgrid, dim3(AHF_BLOCK), 0, c->st, v, per_f, per_m, zn,
                         l.pmask, l.node_p0, l.qp, descending, l.m2pd, kmax, l.dens, heavy, n_heavy);
    else
      hipLaunchKernelGGL((k_gather_full<AHF_FULL_CAP_SMALL, true>), fgrid, dim3(AHF_BLOCK), 0, c->st, v, per_f, per_m,
                         zn, l.pmask, l.node_p0, l.qp, descending, l.m2pd, kmax, l.dens, heavy, n_heavy);
  } else if (dense)
    hipLaunchKernelGGL(k_gather_src, grid, dim3(AHF_BLOCK), 0, c->st, v, tord, per_xcd, l.pmask, l.node_p0, l.qp,
                       descending, l.m2pd, kmax, l.dens, heavy, n_heavy);
  else if ((uint64_t)(n_ent > 0 ? n_ent : 1) * sizeof(ahf_w9) < ((uint64_t)1 << 32) &&
           c->gather_mode != AHFGPU_GATHER_FLAT_WIDE)
    hipLaunchKernelGGL(k_gather_light<true>, grid, dim3(AHF_BLOCK), 0, c->st, v, tord, per_xcd, l.pmask, l.node_p0,
                       l.W, descending, kmax, l.dens, heavy, n_heavy);
  else
    hipLaunchKernelGGL(k_gather_light<false>, grid, dim3(AHF_BLOCK), 0, c->st, v, tord, per_xcd, l.pmask, l.node_p0,
                       l.W, descending, kmax, l.dens, heavy, n_heavy);
  if (timed) c->timer_end(e1, TIMER_GATHER, 12.0 * (double)n_ent + 13.0 * (double)nn);
  hipEvent_t e2 = timed ? c->timer_begin() : nullptr;
  hipLaunchKernelGGL(k_gather_heavy, dim3(AHF_HEAVY_BLOCKS), dim3(AHF_HEAVY_BS), 0, c->st, v, l.pmask, l.node_p0, l.qp,
                     descending, l.m2pd, l.dens, heavy, n_heavy);
  if (timed) c->timer_end(e2, TIMER_HEAVY, 0.0);
  return 0;
}

/* TSC deposit of one level over its n_ent bucket entries in AHF's exact
 * order (even levels walk their lists from the tail of each bucket, odd
 * levels from the head) */
static int deposit_level(ahfgpu_ctx *c, DevLevel &l, int level_index, int64_t n_ent)
{
  const int64_t nn = 8 * l.n_oct;
  if (!l.pmask) {
    l.pmask = c->arena.get<uint32_t>(nn);
    if (!l.pmask) return c->fail(AHFGPU_ENOMEM, "device arena exhausted (pmask, level %d)", level_index);
    level_view v = make_view(l);
    LAUNCH(k_pmask, l.n_oct, v, l.pmask, (uint8_t *)nullptr);
  }
  if (gather_level(c, l, n_ent, (level_index % 2) == 0, true))
    return c->fail(AHFGPU_ENOMEM, "device arena exhausted (deposit, level %d)", level_index);
  return 0;
}

static int build_domain(ahfgpu_ctx *c, DevLevel &d)
{
  const int64_t L = c->params.L_dom, half = L / 2, no = half * half * half, N = c->N;
  d.L = L;
  d.n_oct = no;
  d.n_row = half * half;
  d.n_plane = half;
  Arena &A = c->arena;
  d.oct_key = A.get<uint64_t>(no);
  d.oct_link = A.get<uint8_t>(no);
  d.nbr = A.get<int32_t>(27 * no);
  d.row_key = A.get<uint64_t>(d.n_row);
  d.row_oct0 = A.get<int32_t>(d.n_row + 1);
  d.row_plane = A.get<int32_t>(d.n_row);
  d.plane_z = A.get<int32_t>(d.n_plane);
  d.plane_row0 = A.get<int32_t>(d.n_plane + 1);
  d.node_p0 = A.get<int64_t>(8 * no + 1);
  uint32_t *k0 = A.get<uint32_t>(N), *v0 = A.get<uint32_t>(N), *k1 = A.get<uint32_t>(N), *v1 = A.get<uint32_t>(N);
  uint32_t *rtmp = A.get<uint32_t>(radix_tmp_u32<uint32_t>(N));
  if (!d.oct_key || !d.oct_link || !d.nbr || !d.row_key || !d.row_oct0 || !d.row_plane || !d.plane_z ||
      !d.plane_row0 || !d.node_p0 || !k0 || !v0 || !k1 || !v1 || !rtmp)
    return c->fail(AHFGPU_ENOMEM, "device arena exhausted (domain)");
  LAUNCH(k_domain_octets, no, half, d.oct_key, d.oct_link, d.nbr);
  if ((half & (half - 1)) == 0) {
    d.tord = A.get<uint32_t>(no);
    if (!d.tord) return c->fail(AHFGPU_ENOMEM, "device arena exhausted (domain)");
    LAUNCH(k_morton_full, no, half, d.tord);
  }
  LAUNCH(k_domain_rows, half * half + 1, half, d.row_key, d.row_oct0, d.row_plane, d.plane_z, d.plane_row0);
  hipEvent_t e0 = c->timer_begin();
  LAUNCH(k_bin_domain, N, c->px, c->py, c->pz, N, L, k0, v0);
  int bits = 1;
  while ((1ll << bits) < 8 * no) bits++;
  const int where = radix_sort<uint32_t, uint32_t>(k0, v0, k1, v1, N, bits, rtmp, c->st);
  d.pnode = where ? k1 : k0;
  d.plist = where ? v1 : v0;
  LAUNCH(k_csr_lower_bound, 8 * no + 1, d.pnode, N, 8 * no, d.node_p0);
  c->timer_end(e0, TIMER_BIN, 28.0 * (double)N);
  d.n_part = N;
  const double dl = (double)L;
  d.m2d = (dl * dl * dl) / (double)N;
  d.m2pd = (dl * dl * dl) / (double)N;
  d.crit = c->params.Nth_dom * d.m2d;
  return deposit_level(c, d, 0, N);
}

/* refine level `ci` into a new level; returns 1 if a level was added,
 * 0 when nothing refines or the new level is rolled back, <0 on error */
static int refine_level(ahfgpu_ctx *c, int ci)
{
  DevLevel &l = c->lev[ci];
  Arena &A = c->arena;
  const int64_t nn = 8 * l.n_oct, nrank = 4 * l.n_row, nplr = 2 * l.n_plane;
  level_view v = make_view(l);
  l.flags = A.get<uint8_t>(nn);
  int64_t *cnt = A.get<int64_t>(nrank + 1);
  int64_t *oct_off = A.get<int64_t>(nrank + 1);
  int32_t *rhas = A.get<int32_t>(nrank + 1);
  int32_t *row_off = A.get<int32_t>(nrank + 1);
  int32_t *phas = A.get<int32_t>(nplr + 1);
  int32_t *plane_off = A.get<int32_t>(nplr + 1);
  int64_t *stmp64 = A.get<int64_t>(scan_tmp_elems(nrank));
  int32_t *stmp32 = A.get<int32_t>(scan_tmp_elems(nrank > nplr ? nrank : nplr));
  if (!l.flags || !cnt || !oct_off || !rhas || !row_off || !phas || !plane_off || !stmp64 || !stmp32)
    return c->fail(AHFGPU_ENOMEM, "device arena exhausted (flags, level %d)", ci);
  hipEvent_t e0 = c->timer_begin();
  LAUNCH(k_flags, l.n_oct, v, l.pmask, l.dens, l.crit - 1.0, l.flags);
  hipMemsetAsync(c->d_anomaly, 0, sizeof(int32_t), c->st);
  LAUNCH(k_refine_rows, nrank, v, l.flags, cnt, c->d_anomaly);
  exclusive_scan<int64_t, int64_t>(cnt, oct_off, nrank, stmp64, c->st);
  LAUNCH(k_nonzero, nrank, cnt, nrank, rhas);
  exclusive_scan<int32_t, int32_t>(rhas, row_off, nrank, stmp32, c->st);
  LAUNCH(k_plane_has, nplr, v, cnt, phas);
  exclusive_scan<int32_t, int32_t>(phas, plane_off, nplr, stmp32, c->st);
  c->timer_end(e0, TIMER_REFINE, 4.0 * (double)nn);
  /* sizes of the new level, and the particle count of this level, in one
   * read-back */
  struct {
    int64_t n_oct, n_part, n_row, n_plane, anomaly;
  } sz;
  hipLaunchKernelGGL(k_sizes, dim3(1), dim3(1), 0, c->st, oct_off + nrank, l.node_p0 + nn, row_off + nrank,
                     plane_off + nplr, c->d_anomaly, c->d_sizes);
  hipMemcpyAsync(c->h_sizes, c->d_sizes, 5 * sizeof(int64_t), hipMemcpyDeviceToHost, c->st);
  if (hipStreamSynchronize(c->st) != hipSuccess)
    return c->fail(AHFGPU_EHIP, "refine sizes: %s", hipGetErrorString(hipGetLastError()));
  memcpy(&sz, c->h_sizes, sizeof(sz));
  l.n_part = sz.n_part;
  if (sz.anomaly)
    return c->fail(AHFGPU_EUNSUP, "level %d: AHF would create an empty x-run here (undefined behaviour)", ci);
  if (sz.n_oct == 0) return 0;
  if (ci + 1 >= AHFGPU_MAX_LEVELS) return c->fail(AHFGPU_EINVAL, "too many levels");
  if (8 * sz.n_oct >= (int64_t)UINT32_MAX) return c->fail(AHFGPU_EINVAL, "level %d: too many nodes", ci + 1);
  DevLevel f;
  f.L = 2 * l.L;
  f.n_oct = sz.n_oct;
  f.n_row = sz.n_row;
  f.n_plane = sz.n_plane;
  const int64_t n2 = f.n_oct, nn2 = 8 * n2, nent = l.n_part;
  f.oct_key = A.get<uint64_t>(n2);
  f.oct_link = A.get<uint8_t>(n2);
  f.oct_parent = A.get<int64_t>(n2);
  f.nbr = A.get<int32_t>(27 * n2);
  f.row_key = A.get<uint64_t>(f.n_row);
  f.row_oct0 = A.get<int32_t>(f.n_row + 1);
  f.row_plane = A.get<int32_t>(f.n_row);
  f.plane_z = A.get<int32_t>(f.n_plane);
  f.plane_row0 = A.get<int32_t>(f.n_plane + 1);
  f.pmask = A.get<uint32_t>(nn2);
  f.node_p0 = A.get<int64_t>(nn2 + 1);
  l.node2oct = A.get<int32_t>(nn);
  l.child = A.get<int8_t>(nent);
  int64_t *fcnt = A.get<int64_t>(nn2);
  uint32_t *fbig = A.get<uint32_t>(n2);
  int64_t *ftmp = A.get<int64_t>(scan_tmp_elems(nn2));
  if (!f.oct_key || !f.oct_link || !f.oct_parent || !f.nbr || !f.row_key || !f.row_oct0 || !f.row_plane ||
      !f.plane_z || !f.plane_row0 || !f.pmask || !f.node_p0 || !l.node2oct || !l.child || !fcnt || !fbig || !ftmp)
    return c->fail(AHFGPU_ENOMEM, "device arena exhausted (level %d)", ci + 1);
  hipEvent_t e1 = c->timer_begin();
  hipMemsetAsync(l.node2oct, 0xFF, (size_t)nn * sizeof(int32_t), c->st);
  LAUNCH(k_compact, nrank, v, l.flags, cnt, oct_off, row_off, plane_off, f.oct_key, f.oct_link, f.oct_parent,
         f.row_key, f.row_oct0, f.row_plane, l.node2oct);
  LAUNCH(k_plane_fill, nplr, v, phas, plane_off, row_off, f.plane_z, f.plane_row0);
  if (l.tord) {
    int32_t *mflag = A.get<int32_t>(nn), *mpos = A.get<int32_t>(nn + 1);
    int32_t *mtmp = A.get<int32_t>(scan_tmp_elems(nn));
    f.tord = A.get<uint32_t>(n2);
    if (!mflag || !mpos || !mtmp || !f.tord) return c->fail(AHFGPU_ENOMEM, "device arena exhausted (level %d)", ci + 1);
    LAUNCH(k_morton_next_flags, nn, l.tord, l.node2oct, nn, mflag);
    exclusive_scan<int32_t, int32_t>(mflag, mpos, nn, mtmp, c->st);
    LAUNCH(k_morton_next_emit, nn, l.tord, l.node2oct, nn, mpos, f.tord);
  }
  hipLaunchKernelGGL(k_set2, dim3(1), dim3(1), 0, c->st, f.row_oct0, f.n_row, (int32_t)f.n_oct, f.plane_row0,
                     f.n_plane, (int32_t)f.n_row);
  LAUNCH(k_nbr_next, 27 * n2, l.nbr, f.oct_parent, l.node2oct, n2, f.nbr);
  level_view fv = make_view(f);
  uint8_t *imask2 = A.get<uint8_t>(n2);
  if (!imask2) return c->fail(AHFGPU_ENOMEM, "device arena exhausted (level %d)", ci + 1);
  LAUNCH(k_pmask, fv.n_oct, fv, f.pmask, imask2);
  c->timer_end(e1, TIMER_BUILD, 150.0 * (double)n2);
  /* relink: child of every entry, then the fine buckets */
  hipEvent_t e2 = c->timer_begin();
  LAUNCH(k_relink_child, nent, nent, l.pnode, l.plist, l.node2oct, l.oct_key, imask2, l.qp, c->px, c->py, c->pz,
         (double)f.L, l.child);
  uint32_t *n_big = (uint32_t *)(c->d_anomaly + 2); /* two counts */
  hipMemsetAsync(n_big, 0, 2 * sizeof(uint32_t), c->st);
  LAUNCH(k_fine_count, n2, f.oct_parent, n2, l.node_p0, l.child, fcnt, fbig, n_big);
  hipLaunchKernelGGL(k_fine_big<false>, dim3(2 * AHF_FINE_BLOCKS), dim3(AHF_FINE_BS), 0, c->st, n2, f.oct_parent,
                     l.node_p0, l.child, l.plist, fbig, n_big, fcnt, nullptr, nullptr, nullptr);
  exclusive_scan<int64_t, int64_t>(fcnt, f.node_p0, nn2, ftmp, c->st);
  /* the fine level keeps at most the coarse level's entries */
  f.plist = A.get<uint32_t>(nent);
  f.pnode = A.get<uint32_t>(nent);
  if (!f.plist || !f.pnode) return c->fail(AHFGPU_ENOMEM, "device arena exhausted (level %d)", ci + 1);
  LAUNCH(k_fine_fill, nent, nent, l.pnode, l.node2oct, l.node_p0, l.child, l.plist, f.node_p0, f.plist, f.pnode);
  hipLaunchKernelGGL(k_fine_big<true>, dim3(2 * AHF_FINE_BLOCKS), dim3(AHF_FINE_BS), 0, c->st, n2, f.oct_parent,
                     l.node_p0, l.child, l.plist, fbig, n_big, nullptr, f.node_p0, f.plist, f.pnode);
  c->timer_end(e2, TIMER_RELINK, 29.0 * (double)nent + 24.0 * (double)nn2);
  /* the particles the fine level keeps: its deposit kernel depends on how
   * many entries each node holds, which is read back only where the coarse
   * level's count (an upper bound) leaves the choice open; the bound then
   * sizes the deposit's records and launches, and the count is read with
   * the next level's sizes */
  const int gm = c->gather_mode;
  const bool full_f = marches(c, f.L, f.n_oct);
  const bool decided = gm == AHFGPU_GATHER_FLAT || gm == AHFGPU_GATHER_FLAT_WIDE || gm == AHFGPU_GATHER_SOURCE || full_f ||
                       nent < AHF_DENSE_ENTRIES_PER_NODE * nn2;
  int64_t nent_f = nent;
  f.n_part = -1;
  if (!decided) {
    hipMemcpyAsync(c->h_sizes + 7, f.node_p0 + nn2, sizeof(int64_t), hipMemcpyDeviceToHost, c->st);
    if (hipStreamSynchronize(c->st) != hipSuccess)
      return c->fail(AHFGPU_EHIP, "level %d relink: %s", ci + 1, hipGetErrorString(hipGetLastError()));
    nent_f = c->h_sizes[7];
    f.n_part = nent_f;
  }
  f.m2d = l.m2d * AHF_CRITMULTI_D;
  f.m2pd = l.m2pd * AHF_CRITMULTI_D;
  f.crit = c->params.Nth_ref * f.m2d;
  int rc = deposit_level(c, f, ci + 1, nent_f);
  if (rc) return rc;
  if (nn2 < AHF_MIN_NNODES) {
    /* relink_back (src/libamr_serial/generate_grids.c:231-238): the fine
     * lists go back to their mothers; keep them for the final lists */
    c->rb = f;
    c->rolled_back = 1;
    return 0;
  }
  c->lev.push_back(f);
  return 1;
}

/* ============================================================== C ABI */

extern "C" int ahfgpu_amr_build(ahfgpu_ctx *c, const ahfgpu_amr_params *p, ahfgpu_amr_info *info)
{
  if (!c || !p) return AHFGPU_EINVAL;
  if (c->N <= 0) return c->fail(AHFGPU_EINVAL, "no particles resident (call ahfgpu_set_particles first)");
  /* octets need an even domain grid; refinement doubles it up to L_max */
  bool lmax_ok = p->L_dom >= 4 && (p->L_dom & 1) == 0 && p->L_max >= p->L_dom && p->L_max % p->L_dom == 0;
  if (lmax_ok) {
    const int64_t r = p->L_max / p->L_dom;
    lmax_ok = (r & (r - 1)) == 0;
  }
  if (!lmax_ok)
    return c->fail(AHFGPU_EINVAL, "need an even L_dom >= 4 and L_max = L_dom * 2^k (got %lld, %lld)",
                   (long long)p->L_dom, (long long)p->L_max);
  if (p->L_max > (1 << 22)) return c->fail(AHFGPU_EINVAL, "L_max above 2^22 is not supported");
  if (c->N >= (int64_t)UINT32_MAX) return c->fail(AHFGPU_EINVAL, "at most 2^32-1 particles");
  if ((int64_t)p->L_dom * p->L_dom * p->L_dom >= ((int64_t)1 << 31))
    return c->fail(AHFGPU_EINVAL, "domain grid too large");
  c->params = *p;
  c->arena.reset();
  c->lev.clear();
  c->rolled_back = 0;
  c->rb = DevLevel();
  c->timers_reset(TIMER_BIN, TIMER_RELINK);
  c->timed.clear();
  c->ev_next = 0;
  hipEventRecord(c->ev_a0, c->st);
  c->lev.push_back(DevLevel());
  int rc = build_domain(c, c->lev[0]);
  if (rc) return rc;
  for (;;) {
    const int ci = (int)c->lev.size() - 1;
    if (c->lev[ci].L == p->L_max) break;
    rc = refine_level(c, ci);
    if (rc < 0) return rc;
    if (rc == 0) break;
  }
  hipEventRecord(c->ev_a1, c->st);
  if (hipStreamSynchronize(c->st) != hipSuccess)
    return c->fail(AHFGPU_EHIP, "amr build: %s", hipGetErrorString(hipGetLastError()));
  for (auto *lv : {&c->lev.back(), &c->rb}) {
    if (lv->n_part < 0 && lv->node_p0) {
      hipMemcpy(&lv->n_part, lv->node_p0 + 8 * lv->n_oct, sizeof(int64_t), hipMemcpyDeviceToHost);
    }
  }
  float ms = 0.f;
  hipEventElapsedTime(&ms, c->ev_a0, c->ev_a1);
  c->amr_ms = ms;
  c->timers_collect();
  c->built = 1;
  if (info) {
    memset(info, 0, sizeof(*info));
    info->n_levels = (int32_t)c->lev.size();
    info->rolled_back = c->rolled_back;
    for (size_t i = 0; i < c->lev.size() && i < AHFGPU_MAX_LEVELS; i++) {
      info->n_nodes[i] = 8 * c->lev[i].n_oct;
      info->n_part[i] = c->lev[i].n_part;
      info->deposits += c->lev[i].n_part;
    }
  }
  return 0;
}

/* ---------------------------------------------------- read back levels */

template <typename T>
static std::vector<T> d2h(const T *d, int64_t n, hipStream_t st)
{
  std::vector<T> h((size_t)(n > 0 ? n : 0));
  if (n > 0) hipMemcpyAsync(h.data(), d, (size_t)n * sizeof(T), hipMemcpyDeviceToHost, st);
  return h;
}

/* the same on the host, for when the device has no room for the scratch */
static int final_lists_host(ahfgpu_ctx *c, int lev, int64_t *list0_out, uint32_t *list_out)
{
  const DevLevel &l = c->lev[lev];
  const int64_t nn = 8 * l.n_oct;
  const bool last = lev == (int)c->lev.size() - 1;
  std::vector<int64_t> p0 = d2h(l.node_p0, nn + 1, c->st);
  std::vector<uint32_t> pl = d2h(l.plist, l.n_part, c->st);
  std::vector<int8_t> ch;
  std::vector<int32_t> n2o;
  std::vector<int64_t> fp0;
  std::vector<uint32_t> fpl;
  const bool moved_info = l.child != nullptr;
  const bool rb = last && c->rolled_back;
  if (moved_info) ch = d2h(l.child, l.n_part, c->st);
  if (rb) {
    n2o = d2h(l.node2oct, nn, c->st);
    fp0 = d2h(c->rb.node_p0, 8 * c->rb.n_oct + 1, c->st);
    fpl = d2h(c->rb.plist, c->rb.n_part, c->st);
  }
  if (hipStreamSynchronize(c->st) != hipSuccess) return c->fail(AHFGPU_EHIP, "read back lists");
  std::vector<int64_t> list0((size_t)nn + 1, 0);
  std::vector<uint32_t> list((size_t)l.n_part);
  const bool desc = (lev % 2) == 0, fdesc = ((lev + 1) % 2) == 0;
  int64_t w = 0;
  for (int64_t n = 0; n < nn; n++) {
    list0[(size_t)n] = w;
    const int64_t a = p0[(size_t)n], b = p0[(size_t)n + 1];
    for (int64_t k = 0; k < b - a; k++) {
      const int64_t q = desc ? b - 1 - k : a + k;
      if (!moved_info || ch[(size_t)q] < 0) list[(size_t)w++] = pl[(size_t)q];
    }
    if (rb && n2o[(size_t)n] >= 0) {
      for (int k = 0; k < 8; k++) {
        const int64_t fn = 8 * (int64_t)n2o[(size_t)n] + k;
        const int64_t f0 = fp0[(size_t)fn], f1 = fp0[(size_t)fn + 1];
        for (int64_t j = 0; j < f1 - f0; j++) list[(size_t)w++] = fpl[(size_t)(fdesc ? f1 - 1 - j : f0 + j)];
      }
    }
  }
  list0[(size_t)nn] = w;
  if (list0_out) memcpy(list0_out, list0.data(), list0.size() * sizeof(int64_t));
  if (list_out) memcpy(list_out, list.data(), (size_t)w * sizeof(uint32_t));
  return 0;
}

/*
 * The final per-node lists: of every node the bucket entries that did not move
 * to the next level, in AHF's list order (backwards on even levels), and behind
 * them what a rolled-back level gives back, octant by octant.  rank[q] is the
 * number of entries before q that stay (NULL: all do), so an entry's place
 * follows from its node's bounds alone: flat passes over entries and nodes,
 * bound by memory (17 B an entry, 24 B a node) and the copy to the host.  A
 * clustered 192^3 box's 9 levels, 7.1 million entries: 0.3 ms and the copies
 * beside some 23 ms for the loop over the nodes on the host.
 */
struct StayFlag {
  int8_t child;
  __device__ operator uint32_t() const { return child < 0 ? 1u : 0u; }
};

__device__ __forceinline__ int64_t list_rank(const uint32_t *rank, int64_t q) { return rank ? (int64_t)rank[q] : q; }

/* rbx: per node the entries that a rolled-back level gives to the nodes before
 * it (NULL: none) */
__global__ void k_list_off(int64_t nn, const int64_t *__restrict__ p0, const uint32_t *__restrict__ rank,
                           const int64_t *__restrict__ rbx, int64_t *__restrict__ list0)
{
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n > nn) return;
  list0[n] = list_rank(rank, p0[n]) + (rbx ? rbx[n] : 0);
}

__global__ void k_list_write(int64_t n_ent, const uint32_t *__restrict__ pnode, const uint32_t *__restrict__ plist,
                             const int64_t *__restrict__ p0, const uint32_t *__restrict__ rank, int desc,
                             const int64_t *__restrict__ list0, uint32_t *__restrict__ list)
{
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n_ent) return;
  const int64_t r = list_rank(rank, q);
  if (rank && (int64_t)rank[q + 1] == r) return;
  const int64_t n = pnode[q];
  list[list0[n] + (desc ? list_rank(rank, p0[n + 1]) - 1 - r : r - list_rank(rank, p0[n]))] = plist[q];
}

/* the entries a rolled-back level gives back to every node, and the mother of
 * each of its octets */
__global__ void k_list_rb_count(int64_t nn, const int32_t *__restrict__ node2oct, const int64_t *__restrict__ fp0,
                                int64_t *__restrict__ cnt, int32_t *__restrict__ mother)
{
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= nn) return;
  const int64_t o = node2oct[n];
  cnt[n] = o >= 0 ? fp0[8 * o + 8] - fp0[8 * o] : 0;
  if (o >= 0) mother[o] = (int32_t)n;
}

__global__ void k_list_rb_write(int64_t n_ent, const uint32_t *__restrict__ fpnode, const uint32_t *__restrict__ fplist,
                                const int64_t *__restrict__ fp0, const int32_t *__restrict__ mother,
                                const int64_t *__restrict__ p0, const uint32_t *__restrict__ rank, int fdesc,
                                const int64_t *__restrict__ list0, uint32_t *__restrict__ list)
{
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n_ent) return;
  const int64_t fn = fpnode[q], n = mother[fn >> 3], f0 = fp0[fn], f1 = fp0[fn + 1];
  const int64_t at = list0[n] + list_rank(rank, p0[n + 1]) - list_rank(rank, p0[n]) + f0 - fp0[fn & ~(int64_t)7];
  list[at + (fdesc ? f1 - 1 - q : q - f0)] = fplist[q];
}

/* entries in the final lists of level `lev` */
static int64_t listed_of(const ahfgpu_ctx *c, int lev)
{
  /* particles that stay on this level (plus any rolled back into it) */
  const DevLevel &l = c->lev[lev];
  const bool last = lev == (int)c->lev.size() - 1;
  return l.n_part - (l.child && !last ? c->lev[lev + 1].n_part : 0);
}

/* final per-node lists of level `lev` in AHF's list order into host memory
 * (8*n_oct+1 and listed_of() words; either may be NULL) */
static int final_lists(ahfgpu_ctx *c, int lev, int64_t *list0, uint32_t *list)
{
  const DevLevel &l = c->lev[lev], &f = c->rb;
  const int64_t nn = 8 * l.n_oct, ne = l.n_part, nl = listed_of(c, lev);
  const bool rb = lev == (int)c->lev.size() - 1 && c->rolled_back;
  if (hipSetDevice(c->device) != hipSuccess) return c->fail(AHFGPU_EHIP, "hipSetDevice");
  /* the scratch lies behind the hierarchy and is given back at once */
  Arena &A = c->arena;
  struct Rewind {
    Arena &A;
    Arena::Mark m;
    ~Rewind() { A.rewind(m); }
  } rewind{A, A.mark()};
  const bool ranked = l.child != nullptr;
  int64_t *d0 = A.get<int64_t>(nn + 1), *cnt = nullptr, *rbx = nullptr, *rtmp = nullptr;
  uint32_t *dl = list ? A.get<uint32_t>(nl) : nullptr, *rank = nullptr, *tmp = nullptr;
  int32_t *mother = nullptr;
  bool ok = d0 && (dl || !list);
  if (ranked) {
    rank = A.get<uint32_t>(ne + 1);
    tmp = A.get<uint32_t>(scan_tmp_elems(ne));
    ok = ok && rank && tmp;
  }
  if (rb) {
    cnt = A.get<int64_t>(nn);
    rbx = A.get<int64_t>(nn + 1);
    rtmp = A.get<int64_t>(scan_tmp_elems(nn));
    mother = A.get<int32_t>(f.n_oct);
    ok = ok && cnt && rbx && rtmp && mother;
  }
  if (!ok) return final_lists_host(c, lev, list0, list);
  if (ranked) exclusive_scan<StayFlag, uint32_t>((const StayFlag *)l.child, rank, ne, tmp, c->st);
  if (rb) {
    LAUNCH(k_list_rb_count, nn, nn, l.node2oct, f.node_p0, cnt, mother);
    exclusive_scan<int64_t, int64_t>(cnt, rbx, nn, rtmp, c->st);
  }
  LAUNCH(k_list_off, nn + 1, nn, l.node_p0, rank, rbx, d0);
  if (list && ne > 0)
    LAUNCH(k_list_write, ne, ne, l.pnode, l.plist, l.node_p0, rank, lev % 2 == 0 ? 1 : 0, d0, dl);
  if (list && rb && f.n_part > 0)
    LAUNCH(k_list_rb_write, f.n_part, f.n_part, f.pnode, f.plist, f.node_p0, mother, l.node_p0, rank,
           (lev + 1) % 2 == 0 ? 1 : 0, d0, dl);
  if (list0) hipMemcpyAsync(list0, d0, (size_t)(nn + 1) * sizeof(int64_t), hipMemcpyDeviceToHost, c->st);
  if (list && nl > 0) hipMemcpyAsync(list, dl, (size_t)nl * sizeof(uint32_t), hipMemcpyDeviceToHost, c->st);
  if (hipStreamSynchronize(c->st) != hipSuccess) return c->fail(AHFGPU_EHIP, "read back lists");
  return 0;
}

extern "C" int ahfgpu_amr_level_sizes(ahfgpu_ctx *c, int lev, int64_t *L, int64_t *n_oct, int64_t *n_listed,
                                      double *critdens, double *m2pd)
{
  if (!c || !c->built || lev < 0 || lev >= (int)c->lev.size()) return AHFGPU_EINVAL;
  const DevLevel &l = c->lev[lev];
  if (L) *L = l.L;
  if (n_oct) *n_oct = l.n_oct;
  if (n_listed) *n_listed = listed_of(c, lev);
  if (critdens) *critdens = l.crit;
  if (m2pd) *m2pd = l.m2pd;
  return 0;
}

extern "C" int ahfgpu_amr_level_copy(ahfgpu_ctx *c, int lev, uint64_t *oct_key, uint8_t *oct_link, float *dens,
                                     int64_t *list0, uint32_t *list)
{
  if (!c || !c->built || lev < 0 || lev >= (int)c->lev.size()) return AHFGPU_EINVAL;
  const DevLevel &l = c->lev[lev];
  if (oct_key) hipMemcpyAsync(oct_key, l.oct_key, (size_t)l.n_oct * 8, hipMemcpyDeviceToHost, c->st);
  if (oct_link) hipMemcpyAsync(oct_link, l.oct_link, (size_t)l.n_oct, hipMemcpyDeviceToHost, c->st);
  if (dens) hipMemcpyAsync(dens, l.dens, (size_t)l.n_oct * 8 * 4, hipMemcpyDeviceToHost, c->st);
  if (hipStreamSynchronize(c->st) != hipSuccess) return c->fail(AHFGPU_EHIP, "level copy");
  if (list0 || list) return final_lists(c, lev, list0, list);
  return 0;
}

extern "C" int ahfgpu_amr_dump(ahfgpu_ctx *c, const char *path)
{
  if (!c || !c->built || !path) return AHFGPU_EINVAL;
  const int nl = (int)c->lev.size();
  std::vector<host_level> hl((size_t)nl);
  std::vector<std::vector<uint64_t>> keys((size_t)nl);
  std::vector<std::vector<uint8_t>> links((size_t)nl);
  std::vector<std::vector<float>> dens((size_t)nl);
  std::vector<std::vector<int64_t>> l0((size_t)nl);
  std::vector<std::vector<uint32_t>> li((size_t)nl);
  for (int i = 0; i < nl; i++) {
    const DevLevel &l = c->lev[i];
    keys[(size_t)i] = d2h(l.oct_key, l.n_oct, c->st);
    links[(size_t)i] = d2h(l.oct_link, l.n_oct, c->st);
    dens[(size_t)i] = d2h(l.dens, 8 * l.n_oct, c->st);
    l0[(size_t)i].resize((size_t)(8 * l.n_oct + 1));
    li[(size_t)i].resize((size_t)listed_of(c, i));
    int rc = final_lists(c, i, l0[(size_t)i].data(), li[(size_t)i].data());
    if (rc) return rc;
    host_level &h = hl[(size_t)i];
    memset(&h, 0, sizeof(h));
    h.L = l.L;
    h.n_oct = l.n_oct;
    h.critdens = l.crit;
    h.masstopartdens = l.m2pd;
    h.size_no_nodes = (uint64_t)(8 * l.n_oct);
    h.size_no_part = (uint64_t)l.n_part;
    h.oct_key = keys[(size_t)i].data();
    h.oct_link = links[(size_t)i].data();
    h.dens = dens[(size_t)i].data();
    h.list0 = l0[(size_t)i].data();
    h.list = li[(size_t)i].data();
  }
  return hierarchy_dump(path, hl.data(), nl) ? c->fail(AHFGPU_EIO, "cannot write %s", path) : 0;
}

/* ------------------------------------------------ standalone deposit */

extern "C" int ahfgpu_deposit_level(ahfgpu_ctx *c, int64_t L, const uint64_t *oct_key, const uint8_t *oct_link,
                                    int64_t n_oct, const int64_t *list0, const uint32_t *list, double m2pd,
                                    float *dens_out)
{
  if (!c || !oct_key || !oct_link || !list0 || n_oct <= 0 || L < 4 || (L & 1)) return AHFGPU_EINVAL;
  if (c->N <= 0) return c->fail(AHFGPU_EINVAL, "no particles resident");
  if (hipSetDevice(c->device) != hipSuccess) return c->fail(AHFGPU_EHIP, "hipSetDevice");
  const int64_t nn = 8 * n_oct, ne = list0[nn], half = L / 2;
  for (int64_t i = 1; i < n_oct; i++)
    if (oct_key[i] <= oct_key[i - 1]) return c->fail(AHFGPU_EINVAL, "octet keys must be strictly increasing");
  for (int64_t q = 0; q < ne; q++)
    if ((int64_t)list[q] >= c->N) return c->fail(AHFGPU_EINVAL, "list entry beyond the resident particles");
  /* rows and planes of the octets */
  std::vector<uint64_t> rkey;
  std::vector<int32_t> roct0, rplane, pz, prow0;
  for (int64_t i = 0; i < n_oct; i++) {
    const uint64_t k = oct_key[i];
    const bool new_row = i == 0 || ahf_ky(k) != ahf_ky(oct_key[i - 1]) || ahf_kz(k) != ahf_kz(oct_key[i - 1]);
    if (!new_row) continue;
    if (i == 0 || ahf_kz(k) != ahf_kz(oct_key[i - 1])) {
      pz.push_back((int32_t)ahf_kz(k));
      prow0.push_back((int32_t)rkey.size());
    }
    rkey.push_back((uint64_t)ahf_ky(k) | ((uint64_t)ahf_kz(k) << AHF_KEY_BITS));
    roct0.push_back((int32_t)i);
    rplane.push_back((int32_t)pz.size() - 1);
  }
  roct0.push_back((int32_t)n_oct);
  prow0.push_back((int32_t)rkey.size());
  std::vector<uint32_t> pnode((size_t)(ne > 0 ? ne : 1));
  for (int64_t n = 0; n < nn; n++)
    for (int64_t q = list0[n]; q < list0[n + 1]; q++) pnode[(size_t)q] = (uint32_t)n;
  c->arena.reset();
  c->lev.clear();
  c->built = 0;
  Arena &A = c->arena;
  DevLevel l;
  l.L = L;
  l.n_oct = n_oct;
  l.n_row = (int64_t)rkey.size();
  l.n_plane = (int64_t)pz.size();
  l.oct_key = A.get<uint64_t>(n_oct);
  l.oct_link = A.get<uint8_t>(n_oct);
  l.nbr = A.get<int32_t>(27 * n_oct);
  l.row_key = A.get<uint64_t>(l.n_row);
  l.row_oct0 = A.get<int32_t>(l.n_row + 1);
  l.row_plane = A.get<int32_t>(l.n_row);
  l.plane_z = A.get<int32_t>(l.n_plane);
  l.plane_row0 = A.get<int32_t>(l.n_plane + 1);
  l.node_p0 = A.get<int64_t>(nn + 1);
  l.plist = A.get<uint32_t>(ne);
  l.pnode = A.get<uint32_t>(ne);
  if (!l.oct_key || !l.oct_link || !l.nbr || !l.row_key || !l.row_oct0 || !l.row_plane || !l.plane_z ||
      !l.plane_row0 || !l.node_p0 || !l.plist || !l.pnode)
    return c->fail(AHFGPU_ENOMEM, "device arena exhausted (deposit)");
  hipMemcpyAsync(l.oct_key, oct_key, (size_t)n_oct * 8, hipMemcpyHostToDevice, c->st);
  hipMemcpyAsync(l.oct_link, oct_link, (size_t)n_oct, hipMemcpyHostToDevice, c->st);
  hipMemcpyAsync(l.row_key, rkey.data(), rkey.size() * 8, hipMemcpyHostToDevice, c->st);
  hipMemcpyAsync(l.row_oct0, roct0.data(), roct0.size() * 4, hipMemcpyHostToDevice, c->st);
  hipMemcpyAsync(l.row_plane, rplane.data(), rplane.size() * 4, hipMemcpyHostToDevice, c->st);
  hipMemcpyAsync(l.plane_z, pz.data(), pz.size() * 4, hipMemcpyHostToDevice, c->st);
  hipMemcpyAsync(l.plane_row0, prow0.data(), prow0.size() * 4, hipMemcpyHostToDevice, c->st);
  hipMemcpyAsync(l.node_p0, list0, (size_t)(nn + 1) * 8, hipMemcpyHostToDevice, c->st);
  if (ne > 0) {
    hipMemcpyAsync(l.plist, list, (size_t)ne * 4, hipMemcpyHostToDevice, c->st);
    hipMemcpyAsync(l.pnode, pnode.data(), (size_t)ne * 4, hipMemcpyHostToDevice, c->st);
  }
  LAUNCH(k_nbr_search, 27 * n_oct, l.oct_key, n_oct, half, l.nbr);
  l.m2pd = m2pd;
  /* buckets hold the lists in list order: walk them forwards */
  level_view v = make_view(l);
  l.pmask = A.get<uint32_t>(nn);
  if (!l.pmask) return c->fail(AHFGPU_ENOMEM, "device arena exhausted (deposit)");
  LAUNCH(k_pmask, l.n_oct, v, l.pmask, (uint8_t *)nullptr);
  if (gather_level(c, l, ne, 0, false)) return c->fail(AHFGPU_ENOMEM, "device arena exhausted (deposit)");
  if (dens_out) hipMemcpyAsync(dens_out, l.dens, (size_t)nn * 4, hipMemcpyDeviceToHost, c->st);
  if (hipStreamSynchronize(c->st) != hipSuccess)
    return c->fail(AHFGPU_EHIP, "deposit: %s", hipGetErrorString(hipGetLastError()));
  return 0;
}
