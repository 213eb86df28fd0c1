// Device helpers of neighbour selection (interp/grps.py:141-247,
// pyx:811-890), shared by the standalone selection kernels (spk_neb.hip)
// and the neighbourhood interpolation path (spk_nebk.hip).
#pragma once

#include "spk_internal.h"

namespace spk {

// Strict order on (distance, station index): equal distances are ordered
// by index.
__device__ inline bool lex_less(double a, int ia, double b, int ib) {
  return (a < b) || (a == b && ia < ib);
}

// Wave-wide arg-min of (d, i) pairs; every lane returns the winner.
__device__ inline void wave_argmin(double &d, int &i) {
  for (int off = 32; off > 0; off >>= 1) {
    const double od = __shfl_xor(d, off, 64);
    const int oi = __shfl_xor(i, off, 64);
    if (lex_less(od, oi, d, i)) {
      d = od;
      i = oi;
    }
  }
}

// Angular sector of station (rx, ry) seen from (x, y), pyx:850-868.
__device__ inline long long pie_of(double x, double y, double rx, double ry,
                                   long long n_pies) {
  const double two_pi = 2.0 * kPi;
  const double xd = rx - x, yd = ry - y;
  double ang;
  if (!(xd != 0.0)) {
    ang = 0.0;
  } else {
    ang = atan(yd / xd);
    if (xd < 0 && yd > 0)
      ang = kPi + ang;
    else if (xd < 0 && yd < 0)
      ang = kPi + ang;
    else if (xd > 0 && yd < 0)
      ang = two_pi + ang;
  }
  return (long long)(ang * (double)n_pies / two_pi);
}

// LDS of pie_select for n stations, n_pies sectors and k selections.
__host__ __device__ inline size_t pie_lds_bytes(int n, int n_pies, int k) {
  return (size_t)(n + 2 * n_pies) * 8 + (size_t)(n + 2 * n_pies + k) * 4;
}

// pie for one destination point, run by one 64-thread workgroup: every
// station gets its distance rank inside its angular sector, stations are
// taken rank by rank, nearest first within a rank (interp/grps.py:168-247
// with min_dist_thresh = -1, pyx:846-889).  xy(j) returns station j's
// coordinates.  smem holds pie_lds_bytes(n, n_pies, k), which limits n to
// 16-bit indices.  Writes the first min(k, ranked) selections to sel (LDS,
// selection order) and returns how many were written; a sector index outside
// [0, n_pies) sets bit 1 of bad.
//
// The stations are listed by sector first; a rank then takes one search per
// sector, each by as many lanes as fit side by side (8 sectors: 8 lanes and 3
// steps of reduction each), and the rank's stations find their places by
// counting.  Searching all stations once per sector and rank with the whole
// wavefront, and sorting on one lane, took 5 000 vector instructions for 24 of
// 300 stations in 8 sectors.
template <typename XY>
__device__ int pie_select(int lane, double x, double y, int n, int k,
                          int n_pies, XY xy, char *smem, int **sel_out,
                          int *bad) {
  double *sd = (double *)smem;         // [n]
  int *beg = (int *)(sd + n);          // [n_pies] a sector's first entry
  int *end = beg + n_pies;             // [n_pies] and the one after its last
  double *cand_d = (double *)(end + n_pies);  // [n_pies]
  int *cur = (int *)(cand_d + n_pies);        // [n_pies] last station taken
  int *sel = cur + n_pies;                    // [k]
  int *cand = sel + k;                        // [n_pies]
  unsigned short *sp = (unsigned short *)(cand + n_pies);  // [n] sector
  unsigned short *by = sp + n;                // [n] stations by sector
  *sel_out = sel;
  for (int p = lane; p < n_pies; p += 64) {
    cand[p] = 0;
    cur[p] = -1;
  }
  __syncthreads();
  for (int j = lane; j < n; j += 64) {
    const double2 r = xy(j);
    sd[j] = dist2(x, y, r.x, r.y);
    const long long p = pie_of(x, y, r.x, r.y, n_pies);
    if (p < 0 || p >= n_pies) atomicOr(bad, 1);
    const int q = (int)min(max(p, 0ll), (long long)n_pies - 1);
    sp[j] = (unsigned short)q;
    atomicAdd(&cand[q], 1);
  }
  __syncthreads();
  int base = 0;
  for (int p0 = 0; p0 < n_pies; p0 += 64) {
    const int p = p0 + lane;
    const int v = p < n_pies ? cand[p] : 0;
    int sum = v;
    for (int off = 1; off < 64; off <<= 1) {
      const int u = __shfl_up(sum, off, 64);
      if (lane >= off) sum += u;
    }
    if (p < n_pies) beg[p] = end[p] = base + sum - v;
    base += __shfl(sum, 63, 64);
  }
  __syncthreads();
  for (int j = lane; j < n; j += 64)
    by[atomicAdd(&end[sp[j]], 1)] = (unsigned short)j;
  __syncthreads();
  int width = 64;
  while (width > 1 && width * n_pies > 64) width >>= 1;
  const int at = lane & (width - 1), mine = lane / width, step = 64 / width;
  int nsel = 0;
  while (nsel < k) {
    int ncand = 0;
    for (int p0 = 0; p0 < n_pies; p0 += step) {
      const int p = p0 + mine;
      double bd = INFINITY;
      int bi = 0x7fffffff;
      if (p < n_pies) {
        const int pi = cur[p];
        const double pd = pi < 0 ? -INFINITY : sd[pi];
        for (int e = beg[p] + at; e < end[p]; e += width) {
          const int j = by[e];
          const double d = sd[j];
          if (lex_less(pd, pi, d, j) && lex_less(d, j, bd, bi)) {
            bd = d;
            bi = j;
          }
        }
      }
      for (int off = width >> 1; off > 0; off >>= 1) {
        const double od = __shfl_xor(bd, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        if (lex_less(od, oi, bd, bi)) {
          bd = od;
          bi = oi;
        }
      }
      const bool first = p < n_pies && at == 0;
      if (first) {
        cand[p] = bi;
        cand_d[p] = bd;
        if (bi != 0x7fffffff) cur[p] = bi;
      }
      ncand += __popcll(__ballot(first && bi != 0x7fffffff));
    }
    if (ncand == 0) break;
    __syncthreads();
    // this rank's stations by (distance, index); sectors without one are last
    for (int a = lane; a < n_pies; a += 64) {
      const double ad = cand_d[a];
      const int ai = cand[a];
      int rank = nsel;
      for (int b = 0; b < n_pies; ++b)
        rank += lex_less(cand_d[b], cand[b], ad, ai);
      if (ai != 0x7fffffff && rank < k) sel[rank] = ai;
    }
    nsel += ncand;
    __syncthreads();
  }
  return min(nsel, k);
}

}  // namespace spk
