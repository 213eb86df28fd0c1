// Variogram estimation and fitting for many steps at once
// (variograms/vgs.py:20-870, variograms/fitvgs.py:143-290).
//
//  spk_vgfit_pairs_dev : all station pairs (i > j) sorted by distance, once
//                        per station set (stable radix sort: equal distances
//                        keep the reference's generation order, i then j)
//  spk_vgfit_evg_dev   : per step, the pairs whose two stations have a
//                        value, the mdr distance clip (vgs.py:597-659) and
//                        bins of nk consecutive pairs with the robust or
//                        classic estimator (vgs.py:399-431, 495-520)
//  spk_vgfit_de_dev    : differential evolution (best1bin, dither
//                        U(0.5, 1) per generation, CR 0.7, Latin-hypercube
//                        start, stop when std(E) <= tol |mean(E)|) of every
//                        (step, candidate model) pair over the whole
//                        device; the objective is vgs.py:661-678 without
//                        weights.
#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "spk_internal.h"

namespace spk {

// ---- pairs ---------------------------------------------------------------
__global__ void k_pair_keys(const double *__restrict__ x,
                            const double *__restrict__ y, int64_t N,
                            unsigned long long *__restrict__ key,
                            int64_t *__restrict__ val) {
  const int64_t M = N * (N - 1) / 2;
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < M;
       k += (int64_t)gridDim.x * blockDim.x) {
    // k = i (i - 1) / 2 + j, 0 <= j < i
    int64_t i = (int64_t)floor((1.0 + sqrt(1.0 + 8.0 * (double)k)) * 0.5);
    while (i * (i - 1) / 2 > k) --i;
    while ((i + 1) * i / 2 <= k) ++i;
    const int64_t j = k - i * (i - 1) / 2;
    // vgs.py:327-329: sqrt((x_i - x_j)^2 + (y_i - y_j)^2)
    const double dx = x[i] - x[j], dy = y[i] - y[j];
    double d;
    {
#pragma clang fp contract(off)
      d = sqrt(dx * dx + dy * dy);
    }
    key[k] = __double_as_longlong(d);  // d >= 0: bit order == value order
    val[k] = k;
  }
}

__global__ void k_pair_unpack(const unsigned long long *__restrict__ key,
                              const int64_t *__restrict__ val, int64_t M,
                              int32_t *__restrict__ pi, int32_t *__restrict__ pj,
                              double *__restrict__ pd) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < M;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t k = val[e];
    int64_t i = (int64_t)floor((1.0 + sqrt(1.0 + 8.0 * (double)k)) * 0.5);
    while (i * (i - 1) / 2 > k) --i;
    while ((i + 1) * i / 2 <= k) ++i;
    pi[e] = (int32_t)i;
    pj[e] = (int32_t)(k - i * (i - 1) / 2);
    pd[e] = __longlong_as_double((long long)key[e]);
  }
}

// ---- empirical variograms ----------------------------------------------------
// list: per-step scratch of M int32 (indices into the sorted pair arrays of
// the step's active pairs, in their order).  Written by (chunk, step)
// workgroups in three passes: counts per chunk of kEvgChunk pairs, their
// exclusive scan, then the list; the distance clip and the bins follow.
// One workgroup per step that walked all pairs by itself took 7.2 ms for 24
// steps of 1 500 stations (1.1 million pairs), bound by its serial chain of
// loads; this split takes 0.56 ms.  Steps of few pairs take all passes in one
// workgroup (k_evg_small).
constexpr int kEvgChunk = 4096;

// Active pairs of one chunk: bit u of the result is set when pair
// b0 + tid + 256 u has both values.
__device__ inline unsigned evg_active(const int32_t *pi, const int32_t *pj,
                                      const double *z, int64_t b0, int64_t M) {
  unsigned m = 0;
#pragma unroll
  for (int u = 0; u < kEvgChunk / 256; ++u) {
    const int64_t e = b0 + threadIdx.x + 256 * u;
    if (e < M && !isnan(z[pi[e]]) && !isnan(z[pj[e]])) m |= 1u << u;
  }
  return m;
}

// grid (chunks, steps): cnt[step][chunk]
__global__ __launch_bounds__(256) void k_evg_count(
    const int32_t *__restrict__ pi, const int32_t *__restrict__ pj, int64_t M,
    const double *__restrict__ vals, int64_t N, int64_t *__restrict__ cnt) {
  const double *z = vals + (int64_t)blockIdx.y * N;
  int c = __popc(evg_active(pi, pj, z, (int64_t)blockIdx.x * kEvgChunk, M));
  for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
  __shared__ int w[4];
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0)
    cnt[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] =
        w[0] + w[1] + w[2] + w[3];
}

// One workgroup per step: cnt becomes the chunks' start positions,
// act[step] the number of active pairs.
__global__ __launch_bounds__(256) void k_evg_scan(int64_t *__restrict__ cnt,
                                                  int nchunk,
                                                  int64_t *__restrict__ act) {
  int64_t *c = cnt + (int64_t)blockIdx.x * nchunk;
  __shared__ int64_t sh[256];
  int64_t base = 0;
  for (int k0 = 0; k0 < nchunk; k0 += 256) {
    const int k = k0 + (int)threadIdx.x;
    const int64_t v = k < nchunk ? c[k] : 0;
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int w = 1; w < 256; w <<= 1) {
      const int64_t o = (int)threadIdx.x >= w ? sh[threadIdx.x - w] : 0;
      __syncthreads();
      sh[threadIdx.x] += o;
      __syncthreads();
    }
    if (k < nchunk) c[k] = base + sh[threadIdx.x] - v;
    base += sh[255];
    __syncthreads();
  }
  if (threadIdx.x == 0) act[blockIdx.x] = base;
}

// The chunk's active pairs in their order, from list[base] on, by the
// workgroup; returns how many.
__device__ inline int evg_list(const int32_t *pi, const int32_t *pj,
                               const double *z, int64_t b0, int64_t M,
                               int64_t base, int32_t *L) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned m = evg_active(pi, pj, z, b0, M);
  __shared__ int wcnt[kEvgChunk / 64];  // active pairs per run of 64
  __shared__ int total;
#pragma unroll
  for (int u = 0; u < kEvgChunk / 256; ++u) {
    const unsigned long long bm = __ballot((m >> u) & 1u);
    if (lane == 0) wcnt[u * 4 + wave] = __popcll(bm);
  }
  __syncthreads();
  if (threadIdx.x < 64) {  // exclusive scan of the 64 runs
    const int v = wcnt[lane];
    int x = v;
    for (int w = 1; w < 64; w <<= 1) {
      const int o = __shfl_up(x, w, 64);
      if (lane >= w) x += o;
    }
    wcnt[lane] = x - v;
    if (lane == 63) total = x;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kEvgChunk / 256; ++u) {
    const bool act = (m >> u) & 1u;
    const unsigned long long bm = __ballot(act);
    if (act)
      L[base + wcnt[u * 4 + wave] + __popcll(bm & ((1ull << lane) - 1ull))] =
          (int32_t)(b0 + threadIdx.x + 256 * u);
  }
  return total;
}

// grid (chunks, steps)
__global__ __launch_bounds__(256) void k_evg_list(
    const int32_t *__restrict__ pi, const int32_t *__restrict__ pj, int64_t M,
    const double *__restrict__ vals, int64_t N,
    const int64_t *__restrict__ cnt, int32_t *__restrict__ list) {
  evg_list(pi, pj, vals + (int64_t)blockIdx.y * N,
           (int64_t)blockIdx.x * kEvgChunk, M,
           cnt[(int64_t)blockIdx.y * gridDim.x + blockIdx.x],
           list + (int64_t)blockIdx.y * M);
}

// First position p in [0, hi) of a step's ascending active distances with
// d > v (strict) or not d < v, hi if there is none: 64 probes per round, so
// that a million pairs take four dependent loads.  Run by one wave; every
// lane returns the position.
__device__ inline int64_t evg_first(const double *pd, const int32_t *L,
                                    int64_t hi, double v, bool strict) {
  const int lane = threadIdx.x & 63;
  int64_t lo = 0;
  while (lo < hi) {
    // probes lo, lo + st, ..., each below hi or ignored
    const int64_t st = (hi - lo + 63) / 64;
    const int64_t p = lo + st * lane;
    bool t = false;
    if (p < hi) {
      const double d = pd[L[p]];
      t = strict ? d > v : !(d < v);
    }
    const unsigned long long bm = __ballot(t);
    const unsigned long long in = __ballot(p < hi);
    if (bm == 0) {
      // false at every probe: the answer lies after the last one
      lo += st * (__popcll(in) - 1) + 1;
    } else {
      const int f = __ffsll((long long)bm) - 1;
      hi = lo + st * f;  // true there
      if (f > 0) lo += st * (f - 1) + 1;
    }
  }
  return lo;
}

// The distance clip (vgs.py:597-659) of a step with `base` active pairs:
// argmin |d - mdr max| (first occurrence) over their sorted distances.  Run
// by one wave; every lane returns the pairs kept.
__device__ inline int64_t evg_clip(const double *pd, const int32_t *L,
                                   int64_t base, double mdr) {
  if (base <= 0) return base;
  const double act_max = pd[L[base - 1]];
  const double md = act_max * mdr;
  const int64_t lo = evg_first(pd, L, base, md, true);
  int64_t idx;
  if (lo == 0) {
    idx = 0;
  } else if (lo == base) {
    idx = base - 1;
  } else {
    const double da = md - pd[L[lo - 1]], db = pd[L[lo]] - md;
    idx = (da <= db) ? lo - 1 : lo;
  }
  // first occurrence of that distance value
  idx = evg_first(pd, L, idx, pd[L[idx]], false);
  double clip_ul = pd[L[idx]];
  if (!(clip_ul - md > 0)) clip_ul = md;
  // keep d < clip_ul
  return idx != base - 1 ? evg_first(pd, L, base, clip_ul, false) : base;
}
__device__ inline int evg_nbins(int64_t keep, int nk, int max_bins) {
  return (int)min((keep + nk - 1) / nk, (int64_t)max_bins);
}

// One wave per step.  keep[step]: pairs kept.
__global__ __launch_bounds__(64) void k_evg_clip(
    const double *__restrict__ pd, int64_t M, double mdr, int nk,
    int max_bins, const int32_t *__restrict__ list,
    const int64_t *__restrict__ act, int64_t *__restrict__ keep_out,
    int32_t *__restrict__ nbins) {
  const int s = blockIdx.x;
  const int64_t keep = evg_clip(pd, list + (int64_t)s * M, act[s], mdr);
  if (threadIdx.x == 0) {
    keep_out[s] = keep;
    nbins[s] = evg_nbins(keep, nk, max_bins);
  }
}

// Bin b of a step with `keep` kept pairs, summed in their order by one thread.
__device__ inline void evg_bin(const int32_t *pi, const int32_t *pj,
                               const double *pd, const double *z,
                               const int32_t *L, int64_t keep, int nk,
                               int classic, int b, double *bh, double *bg,
                               int32_t *bn) {
  const int64_t p0 = (int64_t)b * nk;
  const int cntb = (int)min((int64_t)nk, keep - p0);
  double sd = 0.0, sr = 0.0;
  for (int q = 0; q < cntb; ++q) {
    const int32_t e = L[p0 + q];
    sd += pd[e];
    sr += sqrt(fabs(z[pi[e]] - z[pj[e]]));
  }
  double g;
  if (!classic) {
    // vgs.py:414-422
    const double t = sr / cntb;
    const double t4 = (t * t) * (t * t);
    g = (t4 / (0.457 + (0.494 / cntb))) / 2.0;
  } else {
    // vgs.py:399-412: median of squared differences (insertion sort)
    double v[64];
    const int c2 = cntb < 64 ? cntb : 64;
    for (int q = 0; q < c2; ++q) {
      const int32_t e = L[p0 + q];
      const double dz = z[pi[e]] - z[pj[e]];
      double key = dz * dz;
      int w2 = q - 1;
      while (w2 >= 0 && v[w2] > key) {
        v[w2 + 1] = v[w2];
        --w2;
      }
      v[w2 + 1] = key;
    }
    g = (c2 & 1) ? v[c2 / 2] : 0.5 * (v[c2 / 2 - 1] + v[c2 / 2]);
  }
  bh[b] = sd / cntb;
  bg[b] = g;
  bn[b] = cntb;
}

// grid (ceil(max bins / 256), steps)
__global__ __launch_bounds__(256) void k_evg_bins(
    const int32_t *__restrict__ pi, const int32_t *__restrict__ pj,
    const double *__restrict__ pd, int64_t M, const double *__restrict__ vals,
    int64_t N, int nk, int classic, int max_bins,
    const int32_t *__restrict__ list, const int64_t *__restrict__ keep,
    const int32_t *__restrict__ nbins, double *__restrict__ bh,
    double *__restrict__ bg, int32_t *__restrict__ bn) {
  const int s = blockIdx.y;
  const int b = blockIdx.x * 256 + threadIdx.x;
  const int64_t o = (int64_t)s * max_bins;
  if (b < nbins[s])
    evg_bin(pi, pj, pd, vals + (int64_t)s * N, list + (int64_t)s * M, keep[s],
            nk, classic, b, bh + o, bg + o, bn + o);
}

// All passes of a step in one workgroup, for few pairs (kEvgSmall chunks): a
// step's passes are then shorter than their launches.  grid (steps)
constexpr int kEvgSmall = 4;
__global__ __launch_bounds__(256) void k_evg_small(
    const int32_t *pi, const int32_t *pj, const double *pd, int64_t M,
    const double *vals, int64_t N, double mdr, int nk, int classic,
    int max_bins, int32_t *list, double *bh, double *bg, int32_t *bn,
    int32_t *nbins) {
  const int s = blockIdx.x;
  const double *z = vals + (int64_t)s * N;
  int32_t *L = list + (int64_t)s * M;
  __shared__ int64_t keep_s;
  int64_t base = 0;
  for (int64_t b0 = 0; b0 < M; b0 += kEvgChunk) {
    base += evg_list(pi, pj, z, b0, M, base, L);
    __syncthreads();  // the chunk's counts are read, its list is written
  }
  if (threadIdx.x < 64) {
    const int64_t keep = evg_clip(pd, L, base, mdr);
    if (threadIdx.x == 0) {
      keep_s = keep;
      nbins[s] = evg_nbins(keep, nk, max_bins);
    }
  }
  __syncthreads();
  const int64_t keep = keep_s, o = (int64_t)s * max_bins;
  const int nb = evg_nbins(keep, nk, max_bins);
  for (int b = threadIdx.x; b < nb; b += 256)
    evg_bin(pi, pj, pd, z, L, keep, nk, classic, b, bh + o, bg + o, bn + o);
}

// ---- differential evolution ----------------------------------------------------
struct Rng {
  unsigned long long s;
  __device__ explicit Rng(unsigned long long seed) : s(seed ? seed : 1ull) {}
  __device__ inline unsigned long long next() {
    // xorshift64*
    s ^= s >> 12;
    s ^= s << 25;
    s ^= s >> 27;
    return s * 2685821657736338717ull;
  }
  __device__ inline double uni() {  // [0, 1)
    return (double)(next() >> 11) * (1.0 / 9007199254740992.0);
  }
};

__device__ inline unsigned long long mix64(unsigned long long x) {
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}

// vgs.py:533-590 fit models (Sph and Lin switch at h > r)
__device__ inline double fit_model(int t, double h, double r, double s) {
  switch (t) {
    case SPK_VG_NUG: return s;
    case SPK_VG_SPH:
      return h > r ? s : s * ((1.5 * h) / r - (h * h * h) / (2.0 * r * r * r));
    case SPK_VG_EXP: return s * (1.0 - exp(-3.0 * (h / r)));
    case SPK_VG_LIN: return h > r ? s : s * (h / r);
    case SPK_VG_GAU: return s * (1.0 - exp(-3.0 * ((h * h) / (r * r))));
    case SPK_VG_POW: return s * pow(h, r);
    case SPK_VG_HOL: {
      if (!(h > 0)) return 0.0;
      const double x = (kPi * h) / r;
      return s * (1.0 - sin(x) / x);
    }
    default: return NAN;
  }
}

constexpr int kDeMaxD = 8;
constexpr int kDeMaxPop = 800;

// Population of a candidate with D parameters: popmul * D^2, at most
// kDeMaxPop (the host sizes the workgroup's LDS with the same function).
__host__ __device__ inline int de_pop(int popmul, int D) {
  const long long p = (long long)popmul * D * D;
  return p < kDeMaxPop ? (int)p : kDeMaxPop;
}

// Members per thread: member i belongs to thread i mod 256, as its k-th
// member with k = i / 256; its energy and its trial's energy stay in that
// thread's registers.
constexpr int kDeOwn = (kDeMaxPop + 255) / 256;

// LDS of one k_de workgroup for populations of up to pcap members with a
// row stride of ds parameters: population and trials (doubles); the
// Latin-hypercube permutation (pcap ints) shares the trials' space.
inline size_t de_lds_bytes(int pcap, int ds) {
  return (size_t)pcap * ds * 2 * sizeof(double);
}

// a[k] = v for a thread's k-th member (static indices keep a in registers)
__device__ inline void set_own(double (&a)[kDeOwn], int k, double v) {
#pragma unroll
  for (int j = 0; j < kDeOwn; ++j)
    if (j == k) a[j] = v;
}

// The parts of an energy's sum: max(64, ceil(bins / 16)) bins each.
constexpr int kDeSplit = 16;
constexpr int kDeMinBins = 64;

__host__ __device__ inline int de_part_bins(int nb) {
  const int l = (nb + kDeSplit - 1) / kDeSplit;
  return l < kDeMinBins ? kDeMinBins : l;
}

// Bounds of component c's (range, sill) of candidate cd (vgs.py:735-757).
__device__ inline void de_bounds(const int32_t *cd, int c, double h0,
                                 double g0, double v, double range_ub,
                                 double *lb, double *ub) {
  if (cd[1 + c] == SPK_VG_POW) {
    lb[0] = 1e-5;
    ub[0] = 2.0;
    lb[1] = 1e-5;
    ub[1] = 2.0 * v;
  } else if (cd[5] && c == 0) {
    lb[0] = ub[0] = h0;
    lb[1] = ub[1] = g0;
  } else {
    lb[0] = h0;
    ub[0] = range_ub;
    lb[1] = 1e-5;
    ub[1] = 2.0 * v;
  }
}

// sum over bins [b0, b1) of the squares of res(h, g)
template <typename F>
__device__ inline double de_sum(const double *__restrict__ h,
                                const double *__restrict__ g, int b0, int b1,
                                F res) {
  double acc = 0.0;
#pragma unroll 4
  for (int b = b0; b < b1; ++b) {
    const double d = res(h[b], g[b]);
    acc = fma(d, d, acc);
  }
  return acc;
}

// The components of a candidate: `others` besides the constant ones (nuggets),
// of which component `one` (of model ty) if it is the only one.
struct DeCand {
  int n, one, others, ty;
};
__device__ inline DeCand de_cand(const int32_t *cd) {
  DeCand q = {cd[0], -1, 0, SPK_VG_NUG};
  for (int c = 0; c < q.n; ++c)
    if (cd[1 + c] != SPK_VG_NUG) {
      q.one = c;
      q.ty = cd[1 + c];
      ++q.others;
    }
  return q;
}

// An energy's share of bins [b0, b1) of a step whose bins are h and g: the
// squared residuals (vgs.py:661-678) of member x between lb and ub (de_bounds,
// in LDS).  Both evolutions below add the same parts in the same order, so that
// a step's result does not depend on which of them takes it.  The model's value
// is rounded before it is subtracted: a step of one bin converges when every
// member meets it to the last bit (about 250 generations; with the residual
// formed in one operation it never did, and took 10 000).
__device__ inline double de_part(const DeCand &dc, const int32_t *cd,
                                 const double *x,
                                 const double *lb, const double *ub,
                                 const double *__restrict__ h,
                                 const double *__restrict__ g, int b0, int b1) {
#pragma clang fp contract(off)
  const int ncomp = dc.n, one = dc.one, others = dc.others, ty = dc.ty;
  double acc;
  double nug = 0.0, rg = 1.0, sl = 0.0;
  auto par = [&](int d) { return fma(x[d], ub[d] - lb[d], lb[d]); };
  for (int c = 0; c < ncomp; ++c) {
    if (cd[1 + c] == SPK_VG_NUG) {
      nug += par(2 * c + 1);
    } else if (c == one) {
      rg = par(2 * c);
      sl = par(2 * c + 1);
    }
  }
  if (others == 0) {
    acc = de_sum(h, g, b0, b1, [&](double, double gb) { return gb - nug; });
  } else if (others == 1 && ty == SPK_VG_EXP) {
    // (the bound keeps a range of zero, -inf, out of exp2_neg)
    const double c = (-3.0 / rg) * kLog2e, top = nug + sl;
    acc = de_sum(h, g, b0, b1, [&](double hb, double gb) {
      return gb - fma(-sl, exp2_neg<false>(fmax(hb * c, -1100.0)), top);
    });
  } else if (others == 1 && ty == SPK_VG_GAU) {
    const double c = (-3.0 / (rg * rg)) * kLog2e, top = nug + sl;
    acc = de_sum(h, g, b0, b1, [&](double hb, double gb) {
      return gb - fma(-sl, exp2_neg<false>(fmax((hb * hb) * c, -1100.0)), top);
    });
  } else if (others == 1 && ty == SPK_VG_SPH) {
    const double c = 1.0 / rg;
    acc = de_sum(h, g, b0, b1, [&](double hb, double gb) {
      const double u = fmin(hb * c, 1.0);  // the sill at h >= r
      return gb - fma(sl, u * fma(u * u, -0.5, 1.5), nug);
    });
  } else {
    acc = 0.0;
    for (int b = b0; b < b1; ++b) {
      const double hb = h[b];
      double y = 0.0;
      for (int c = 0; c < ncomp; ++c)
        y += fit_model(cd[1 + c], hb, par(2 * c), par(2 * c + 1));
      const double r = g[b] - y;
      acc = fma(r, r, acc);
    }
  }
  return acc;
}

__device__ inline double blk_sum(double v, double *red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

// (bv, bi) <- the smaller of (bv, bi) and (ov, oi) by value, then index;
// bi == INT_MAX marks an empty slot
__device__ inline void argmin_take(double &bv, int &bi, double ov, int oi) {
  if (oi != INT_MAX && (bi == INT_MAX || ov < bv || (ov == bv && oi < bi))) {
    bv = ov;
    bi = oi;
  }
}

// Index of the smallest energy of members i < P (each thread holds its own
// members' energies, en[k] of member threadIdx.x + 256 k) over the 256
// threads of the block: the first index among equal values, and NaN
// entries never chosen, which is what the scan
// `bi = 0; for i: if (en[i] < en[bi]) bi = i` returns (that scan keeps 0
// when the energy of member 0 is NaN).  Every thread gets the index and,
// in best, its energy.
__device__ inline int blk_argmin(const double (&en)[kDeOwn], int P,
                                 double *rv, int *ri, double *e0,
                                 double &best) {
  double bv = 0.0;
  int bi = INT_MAX;
#pragma unroll
  for (int k = 0; k < kDeOwn; ++k) {
    const int i = threadIdx.x + 256 * k;
    if (i < P) {
      const double v = en[k];
      if (!isnan(v) && (bi == INT_MAX || v < bv)) {
        bv = v;
        bi = i;
      }
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    const double ov = __shfl_xor(bv, off, 64);
    const int oi = __shfl_xor(bi, off, 64);
    argmin_take(bv, bi, ov, oi);
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    rv[threadIdx.x >> 6] = bv;
    ri[threadIdx.x >> 6] = bi;
  }
  if (threadIdx.x == 0) *e0 = en[0];
  __syncthreads();
  bv = rv[0];
  bi = ri[0];
  for (int w = 1; w < 4; ++w) argmin_take(bv, bi, rv[w], ri[w]);
  if (isnan(*e0) || bi == INT_MAX) {
    best = *e0;
    return 0;
  }
  best = bv;
  return bi;
}

// One workgroup per (step, candidate).  cand[c]: {ncomp, type[4],
// fixed_first}; with fixed_first the first component's (range, sill) are
// pinned to the step's first bin (h0, g0), vgs.py:735-739.
__global__ __launch_bounds__(256, 3) void k_de(
    const double *__restrict__ bh, const double *__restrict__ bg,
    const int32_t *__restrict__ nbins, int max_bins,
    const double *__restrict__ var, const int32_t *__restrict__ cand,
    int ncand, int maxiter, int popmul, double tol, double range_ub,
    unsigned long long seed, const double *__restrict__ init, double spread,
    int pcap, int ds, double *__restrict__ out_par,
    double *__restrict__ out_fun, int32_t *__restrict__ out_nit) {
  const int s = blockIdx.y, ci = blockIdx.x;
  const int tid = threadIdx.x;
  const int32_t *cd = cand + ci * 6;
  const int ncomp = cd[0];
  const int D = 2 * ncomp;
  const int P = de_pop(popmul, D);
  const int nb = nbins[s];
  const double *h = bh + (int64_t)s * max_bins;
  const double *g = bg + (int64_t)s * max_bins;
  // LDS sized by the launch for its largest population (pcap) and
  // parameter count (ds, the row stride), so that small candidates leave
  // room for more workgroups per CU
  extern __shared__ double de_lds[];
  double *pop = de_lds;
  double *trial = pop + (int64_t)pcap * ds;
  int *perm = (int *)trial;  // start only, before the first trial
  __shared__ double lb[kDeMaxD], ub[kDeMaxD];
  __shared__ double red[4];
  __shared__ double redv[4];
  __shared__ int redi[4];
  __shared__ double e0s;
  __shared__ double Fs;
  __shared__ int stop_s;
  double *opar = out_par + ((int64_t)s * ncand + ci) * kDeMaxD;
  if (nb <= 0 || P > pcap || D > ds) {
    if (tid == 0) {
      out_fun[(int64_t)s * ncand + ci] = NAN;
      out_nit[(int64_t)s * ncand + ci] = 0;
    }
    return;
  }
  if (tid == 0)
    for (int c = 0; c < ncomp; ++c)
      de_bounds(cd, c, h[0], g[0], var[s], range_ub, lb + 2 * c, ub + 2 * c);
  Rng rng(mix64(seed ^ mix64(((unsigned long long)s << 20) ^
                             ((unsigned long long)ci << 8) ^ tid)));
  __syncthreads();
  // Latin hypercube start: per dimension a random permutation of P
  // segments plus a uniform offset inside each segment
  for (int d = 0; d < D; ++d) {
    if (tid == 0) {
      for (int i = 0; i < P; ++i) perm[i] = i;
      for (int i = P - 1; i > 0; --i) {
        const int j = (int)(rng.uni() * (i + 1));
        const int t = perm[i];
        perm[i] = perm[j];
        perm[j] = t;
      }
    }
    __syncthreads();
    if (!init) {
      for (int i = tid; i < P; i += 256)
        pop[i * ds + d] = (perm[i] + rng.uni()) / P;
    } else {
      // seeded start: member 0 is the given point; the others stratify a
      // log-box of half-width `spread` around it, clipped to the bounds
      const double w = ub[d] - lb[d];
      const double c = fmin(fmax(init[((int64_t)s * ncand + ci) * kDeMaxD + d],
                                 lb[d]), ub[d]);
      for (int i = tid; i < P; i += 256) {
        double u = 0.0;
        if (w > 0.0) {
          double v = c;
          if (i > 0)
            v = c * exp(spread * (2.0 * (perm[i] + rng.uni()) / P - 1.0));
          v = fmin(fmax(v, lb[d]), ub[d]);
          u = (v - lb[d]) / w;
        }
        pop[i * ds + d] = u;
      }
    }
    __syncthreads();
  }
  const int len = de_part_bins(nb);
  const DeCand dc = de_cand(cd);
  auto energy = [&](const double *x) {
    double e = 0.0;
    for (int b0 = 0; b0 < nb; b0 += len)
      e += de_part(dc, cd, x, lb, ub, h, g, b0, min(nb, b0 + len));
    return e;
  };
  double en[kDeOwn], trial_e[kDeOwn];
#pragma unroll
  for (int k = 0; k < kDeOwn; ++k) en[k] = trial_e[k] = 0.0;
  for (int k = 0; tid + 256 * k < P; ++k) {
    const int i = tid + 256 * k;
    set_own(en, k, energy(&pop[i * ds]));
  }
  __syncthreads();
  int nit = 0;
  double best;
  for (int it = 1; it <= maxiter; ++it) {
    nit = it;
    const int bi = blk_argmin(en, P, redv, redi, &e0s, best);
    if (tid == 0) Fs = 0.5 + 0.5 * rng.uni();
    __syncthreads();
    const double F = Fs;
    // trials and their energies first, selection after (deferred update)
    for (int k = 0; tid + 256 * k < P; ++k) {
      const int i = tid + 256 * k;
      int r0, r1;
      do { r0 = (int)(rng.uni() * P); } while (r0 == i);
      do { r1 = (int)(rng.uni() * P); } while (r1 == i || r1 == r0);
      const int fill = (int)(rng.uni() * D);
      double *tr = &trial[i * ds];
      for (int d = 0; d < D; ++d) {
        double v = pop[i * ds + d];
        if (d == fill || rng.uni() < 0.7) {
          v = pop[bi * ds + d] +
              F * (pop[r0 * ds + d] - pop[r1 * ds + d]);
          if (v < 0.0 || v > 1.0) v = rng.uni();
        }
        tr[d] = v;
      }
      set_own(trial_e, k, energy(tr));
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kDeOwn; ++k) {
      const int i = tid + 256 * k;
      if (i < P && trial_e[k] <= en[k]) {
        en[k] = trial_e[k];
        for (int d = 0; d < D; ++d) pop[i * ds + d] = trial[i * ds + d];
      }
    }
    __syncthreads();
    // convergence: std(E) <= tol * |mean(E)|
    double sm = 0.0;
#pragma unroll
    for (int k = 0; k < kDeOwn; ++k)
      if (tid + 256 * k < P) sm += en[k];
    const double mean = blk_sum(sm, red) / P;
    double sq = 0.0;
#pragma unroll
    for (int k = 0; k < kDeOwn; ++k) {
      if (tid + 256 * k < P) {
        const double dv = en[k] - mean;
        sq += dv * dv;
      }
    }
    const double sd = sqrt(blk_sum(sq, red) / P);
    if (tid == 0) stop_s = (sd <= tol * fabs(mean)) ? 1 : 0;
    __syncthreads();
    if (stop_s) break;
  }
  const int bi = blk_argmin(en, P, redv, redi, &e0s, best);
  if (tid == 0) {
    for (int d = 0; d < kDeMaxD; ++d)
      opar[d] = d < D ? lb[d] + pop[bi * ds + d] * (ub[d] - lb[d]) : 0.0;
    out_fun[(int64_t)s * ncand + ci] = best;
    out_nit[(int64_t)s * ncand + ci] = nit;
  }
}

// ---- differential evolution over the whole device ------------------------------
// The same evolution as k_de, generation by generation in two launches: the
// energies of all candidates' trials over (member groups, bin chunks), then
// one workgroup per candidate that selects, tests convergence and draws the
// next trials.  k_de keeps a candidate on one CU, and its time is the
// largest candidate's: 800 members x 16 000 bins x 2 components of exp() per
// generation, 1 200 ms for a day of 24 steps x 7 candidates with 168 of 256
// CUs in use and most of them early idle.  Spread over the device the same
// day takes 11 ms (energies 9.1, selection and trials 1.3), bound by FP64
// VALU issue: 21 instructions per member and bin for the exponential, 0.2 ms
// per generation of the day's 430 million model values.  The random streams, the order of the draws and the
// selection are k_de's; an energy's sum over bins is taken in kDeSplit
// parts, whose bounds depend on the step's bins only.

// One wave: 64 members of one candidate over one chunk of its step's bins.
// grid (waves / 4, candidates); q = step * ncand + candidate within the
// batch, list (optional) the batch's candidates still evolving.
__global__ __launch_bounds__(256) void k_de_energy(
    const double *__restrict__ bh, const double *__restrict__ bg,
    const int32_t *__restrict__ nbins, int max_bins,
    const double *__restrict__ var, const int32_t *__restrict__ cand,
    int ncand, int popmul, double range_ub, int pcap, int ds,
    const double *__restrict__ mem, const int32_t *__restrict__ list,
    const int32_t *__restrict__ done, double *__restrict__ part) {
  const int q = list ? list[blockIdx.y] : (int)blockIdx.y;
  if (done[q]) return;
  const int s = q / ncand, ci = q - s * ncand;
  const int32_t *cd = cand + ci * 6;
  const int P = de_pop(popmul, 2 * cd[0]);
  const int nb = nbins[s];
  const double *h = bh + (int64_t)s * max_bins;
  const double *g = bg + (int64_t)s * max_bins;
  __shared__ double lb[kDeMaxD], ub[kDeMaxD];
  if ((int)threadIdx.x < cd[0])
    de_bounds(cd, threadIdx.x, h[0], g[0], var[s], range_ub,
              lb + 2 * threadIdx.x, ub + 2 * threadIdx.x);
  __syncthreads();
  const int mgs = (P + 63) / 64;
  const int wv = __builtin_amdgcn_readfirstlane(
      (int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  const int ch = wv / mgs, mg = wv - ch * mgs;
  const int len = de_part_bins(nb);
  const int b0 = ch * len, b1 = min(nb, b0 + len);
  if (ch >= kDeSplit || b0 >= b1) return;
  const int i = mg * 64 + (int)(threadIdx.x & 63);
  const double *x = mem + ((int64_t)q * pcap + min(i, P - 1)) * ds;
  const double acc = de_part(de_cand(cd), cd, x, lb, ub, h, g, b0, b1);
  if (i < P) part[((int64_t)q * kDeSplit + ch) * pcap + i] = acc;
}

// The start population of every candidate of a batch (k_de's
// Latin-hypercube or seeded start); s0: the batch's first step within the
// launch sequence's numbering, which keys the random streams.
__global__ __launch_bounds__(256) void k_de_init(
    const double *__restrict__ bh, const double *__restrict__ bg,
    const int32_t *__restrict__ nbins, int max_bins,
    const double *__restrict__ var, const int32_t *__restrict__ cand,
    int ncand, int popmul, double range_ub, unsigned long long seed, int s0,
    const double *__restrict__ init, double spread, int pcap, int ds,
    double *__restrict__ pop, unsigned long long *__restrict__ rngs,
    int32_t *__restrict__ done, double *__restrict__ out_fun,
    int32_t *__restrict__ out_nit) {
  const int s = blockIdx.y, ci = blockIdx.x, q = s * ncand + ci;
  const int tid = threadIdx.x;
  const int32_t *cd = cand + ci * 6;
  const int D = 2 * cd[0], P = de_pop(popmul, D);
  const bool none = nbins[s] <= 0 || P > pcap || D > ds;
  if (tid == 0) done[q] = none ? 1 : 0;
  if (none) {
    if (tid == 0) {
      out_fun[q] = NAN;
      out_nit[q] = 0;
    }
    return;
  }
  __shared__ int perm[kDeMaxPop];
  Rng rng(mix64(seed ^ mix64(((unsigned long long)(s0 + s) << 20) ^
                             ((unsigned long long)ci << 8) ^ tid)));
  pop += (int64_t)q * pcap * ds;
  for (int d = 0; d < D; ++d) {
    if (tid == 0) {
      for (int i = 0; i < P; ++i) perm[i] = i;
      for (int i = P - 1; i > 0; --i) {
        const int j = (int)(rng.uni() * (i + 1));
        const int t = perm[i];
        perm[i] = perm[j];
        perm[j] = t;
      }
    }
    __syncthreads();
    if (!init) {
      for (int i = tid; i < P; i += 256)
        pop[i * ds + d] = (perm[i] + rng.uni()) / P;
    } else {
      double lb[2], ub[2];
      de_bounds(cd, d >> 1, bh[(int64_t)s * max_bins],
                bg[(int64_t)s * max_bins], var[s], range_ub, lb, ub);
      const double l = lb[d & 1], u1 = ub[d & 1], w = u1 - l;
      const double c = fmin(fmax(init[(int64_t)q * kDeMaxD + d], l), u1);
      for (int i = tid; i < P; i += 256) {
        double u = 0.0;
        if (w > 0.0) {
          double v = c;
          if (i > 0)
            v = c * exp(spread * (2.0 * (perm[i] + rng.uni()) / P - 1.0));
          v = fmin(fmax(v, l), u1);
          u = (v - l) / w;
        }
        pop[i * ds + d] = u;
      }
    }
    __syncthreads();
  }
  rngs[(int64_t)q * 256 + tid] = rng.s;
}

// One workgroup per candidate: takes the energies of generation `it`'s
// trials (0: of the start population), selects, stops the candidate on
// convergence or at maxiter, else draws the trials of generation it + 1.
// The population is staged in LDS (pcap x ds doubles).
__global__ __launch_bounds__(256) void k_de_step(
    const double *__restrict__ bh, const double *__restrict__ bg,
    const int32_t *__restrict__ nbins, int max_bins,
    const double *__restrict__ var, const int32_t *__restrict__ cand,
    int ncand, int it, int maxiter, int popmul, double tol, double range_ub,
    int pcap, int ds, double *__restrict__ pop, double *__restrict__ trial,
    double *__restrict__ energy, const double *__restrict__ part,
    unsigned long long *__restrict__ rngs, const int32_t *__restrict__ list,
    int32_t *__restrict__ done, double *__restrict__ out_par,
    double *__restrict__ out_fun, int32_t *__restrict__ out_nit) {
  const int q = list ? list[blockIdx.x] : (int)blockIdx.x;
  if (done[q]) return;
  const int s = q / ncand, ci = q - s * ncand;
  const int tid = threadIdx.x;
  const int32_t *cd = cand + ci * 6;
  const int D = 2 * cd[0], P = de_pop(popmul, D);
  const int nb = nbins[s];
  const int nch = (nb + de_part_bins(nb) - 1) / de_part_bins(nb);
  extern __shared__ double de_lds[];  // the population
  __shared__ double red[4], redv[4], e0s, Fs;
  __shared__ int redi[4];
  pop += (int64_t)q * pcap * ds;
  trial += (int64_t)q * pcap * ds;
  energy += (int64_t)q * pcap;
  part += (int64_t)q * kDeSplit * pcap;
  double en[kDeOwn];
#pragma unroll
  for (int k = 0; k < kDeOwn; ++k) en[k] = 0.0;
  for (int k = 0; tid + 256 * k < P; ++k) {
    const int i = tid + 256 * k;
    double e = 0.0;
    for (int c = 0; c < nch; ++c) e += part[(int64_t)c * pcap + i];
    const double old = it > 0 ? energy[i] : 0.0;
    const bool take = it == 0 || e <= old;
    const double *src = it > 0 && take ? trial : pop;
    for (int d = 0; d < D; ++d) {
      const double v = src[i * ds + d];
      de_lds[i * ds + d] = v;
      if (it > 0 && take) pop[i * ds + d] = v;
    }
    if (take) energy[i] = e;
    set_own(en, k, take ? e : old);
  }
  __syncthreads();
  bool stop = false;
  if (it > 0) {
    // convergence: std(E) <= tol * |mean(E)|
    double sm = 0.0;
#pragma unroll
    for (int k = 0; k < kDeOwn; ++k)
      if (tid + 256 * k < P) sm += en[k];
    const double mean = blk_sum(sm, red) / P;
    double sq = 0.0;
#pragma unroll
    for (int k = 0; k < kDeOwn; ++k) {
      if (tid + 256 * k < P) {
        const double dv = en[k] - mean;
        sq += dv * dv;
      }
    }
    const double sd = sqrt(blk_sum(sq, red) / P);
    stop = sd <= tol * fabs(mean) || it >= maxiter;
  }
  double best;
  const int bi = blk_argmin(en, P, redv, redi, &e0s, best);
  if (stop) {
    if (tid == 0) {
      for (int c = 0; c < kDeMaxD / 2; ++c) {
        double lb[2] = {0.0, 0.0}, ub[2] = {0.0, 0.0};
        if (c < cd[0])
          de_bounds(cd, c, bh[(int64_t)s * max_bins],
                    bg[(int64_t)s * max_bins], var[s], range_ub, lb, ub);
        for (int e = 0; e < 2; ++e)
          out_par[(int64_t)q * kDeMaxD + 2 * c + e] =
              c < cd[0]
                  ? lb[e] + de_lds[bi * ds + 2 * c + e] * (ub[e] - lb[e])
                  : 0.0;
      }
      out_fun[q] = best;
      out_nit[q] = it;
      done[q] = 1;
    }
    return;
  }
  Rng rng(1);
  rng.s = rngs[(int64_t)q * 256 + tid];
  if (tid == 0) Fs = 0.5 + 0.5 * rng.uni();
  __syncthreads();
  const double F = Fs;
  for (int i = tid; i < P; i += 256) {
    int r0, r1;
    do { r0 = (int)(rng.uni() * P); } while (r0 == i);
    do { r1 = (int)(rng.uni() * P); } while (r1 == i || r1 == r0);
    const int fill = (int)(rng.uni() * D);
    for (int d = 0; d < D; ++d) {
      double v = de_lds[i * ds + d];
      if (d == fill || rng.uni() < 0.7) {
        v = de_lds[bi * ds + d] +
            F * (de_lds[r0 * ds + d] - de_lds[r1 * ds + d]);
        if (v < 0.0 || v > 1.0) v = rng.uni();
      }
      trial[i * ds + d] = v;
    }
  }
  rngs[(int64_t)q * 256 + tid] = rng.s;
}

// ---- spatial order of cells -------------------------------------------------
// Morton (Z-order) keys of the cells' coordinates quantised to 2^20 levels
// per axis over their bounding box; sorting by key makes runs of 64 / 256
// consecutive cells spatially compact tiles.
__global__ void k_bbox_part(const double *__restrict__ x,
                            const double *__restrict__ y, int64_t n,
                            double *__restrict__ part) {
  __shared__ double r[4][256];
  double a = INFINITY, b = -INFINITY, c = INFINITY, d = -INFINITY;
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256) {
    a = fmin(a, x[i]);
    b = fmax(b, x[i]);
    c = fmin(c, y[i]);
    d = fmax(d, y[i]);
  }
  r[0][threadIdx.x] = a;
  r[1][threadIdx.x] = b;
  r[2][threadIdx.x] = c;
  r[3][threadIdx.x] = d;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      r[0][threadIdx.x] = fmin(r[0][threadIdx.x], r[0][threadIdx.x + w]);
      r[1][threadIdx.x] = fmax(r[1][threadIdx.x], r[1][threadIdx.x + w]);
      r[2][threadIdx.x] = fmin(r[2][threadIdx.x], r[2][threadIdx.x + w]);
      r[3][threadIdx.x] = fmax(r[3][threadIdx.x], r[3][threadIdx.x + w]);
    }
    __syncthreads();
  }
  if (threadIdx.x < 4) part[blockIdx.x * 4 + threadIdx.x] = r[threadIdx.x][0];
}

__device__ inline unsigned long long spread_bits(unsigned long long v) {
  v &= 0xffffffffull;
  v = (v | (v << 16)) & 0x0000ffff0000ffffull;
  v = (v | (v << 8)) & 0x00ff00ff00ff00ffull;
  v = (v | (v << 4)) & 0x0f0f0f0f0f0f0f0full;
  v = (v | (v << 2)) & 0x3333333333333333ull;
  v = (v | (v << 1)) & 0x5555555555555555ull;
  return v;
}

__global__ void k_morton(const double *__restrict__ x,
                         const double *__restrict__ y, int64_t n,
                         const double *__restrict__ part, int nparts,
                         unsigned long long *__restrict__ key,
                         int32_t *__restrict__ val) {
  double x0 = INFINITY, x1 = -INFINITY, y0 = INFINITY, y1 = -INFINITY;
  for (int k = 0; k < nparts; ++k) {
    x0 = fmin(x0, part[4 * k]);
    x1 = fmax(x1, part[4 * k + 1]);
    y0 = fmin(y0, part[4 * k + 2]);
    y1 = fmax(y1, part[4 * k + 3]);
  }
  const double span = fmax(fmax(x1 - x0, y1 - y0), 1e-300);
  const double sc = 1048575.0 / span;
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256) {
    double qx = (x[i] - x0) * sc, qy = (y[i] - y0) * sc;
    qx = fmin(fmax(qx, 0.0), 1048575.0);  // NaN coordinates sort first
    qy = fmin(fmax(qy, 0.0), 1048575.0);
    const unsigned long long ix = (unsigned long long)qx;
    const unsigned long long iy = (unsigned long long)qy;
    key[i] = spread_bits(ix) | (spread_bits(iy) << 1);
    val[i] = (int32_t)i;
  }
}

__global__ void k_gather_xy(const double *__restrict__ x,
                            const double *__restrict__ y,
                            const int32_t *__restrict__ perm, int64_t n,
                            double *__restrict__ px, double *__restrict__ py) {
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256) {
    px[i] = x[perm[i]];
    py[i] = y[perm[i]];
  }
}

int cell_order(spk_ctx *ctx, const double *cx, const double *cy, int64_t C,
               int32_t *perm, double *pcx, double *pcy) {
  if (C > INT32_MAX) return set_error(SPK_ESHAPE, "too many cells");
  constexpr int kParts = 256;
  hipStream_t st = ctx->stream;
  double *part;
  unsigned long long *k0, *k1;
  int32_t *v0;
  SPK_TRY(ws_get(ctx, "co_part", kParts * 4 * 8, (void **)&part));
  SPK_TRY(ws_get(ctx, "co_k0", C * 8, (void **)&k0));
  SPK_TRY(ws_get(ctx, "co_k1", C * 8, (void **)&k1));
  SPK_TRY(ws_get(ctx, "co_v0", C * 4, (void **)&v0));
  const unsigned g = (unsigned)std::min<int64_t>(ceil_div(C, 256), 4096);
  hipLaunchKernelGGL(k_bbox_part, dim3(kParts), dim3(256), 0, st, cx, cy, C,
                     part);
  hipLaunchKernelGGL(k_morton, dim3(g), dim3(256), 0, st, cx, cy, C, part,
                     kParts, k0, v0);
  SPK_TRY(check_launch("k_morton"));
  size_t tmp_bytes = 0;
  SPK_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, k0, k1, v0,
                                             perm, (int)C, 0, 40, st));
  void *tmp;
  SPK_TRY(ws_get(ctx, "co_tmp", tmp_bytes, &tmp));
  SPK_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, k0, k1, v0, perm,
                                             (int)C, 0, 40, st));
  hipLaunchKernelGGL(k_gather_xy, dim3(g), dim3(256), 0, st, cx, cy, perm, C,
                     pcx, pcy);
  return check_launch("k_gather_xy");
}

}  // namespace spk

using namespace spk;

extern "C" {

int spk_vgfit_pairs_dev(spk_ctx *ctx, const double *x, const double *y,
                        int64_t N, int32_t *pi, int32_t *pj, double *pd) {
  if (!ctx || !x || !y || !pi || !pj || !pd)
    return set_error(SPK_EARG, "null argument");
  if (N < 2) return set_error(SPK_ESHAPE, "need at least two stations");
  if (N > 46000) return set_error(SPK_ESHAPE, "too many stations for pairs");
  SPK_HIP(hipSetDevice(ctx->device));
  const int64_t M = N * (N - 1) / 2;
  unsigned long long *k0, *k1;
  int64_t *v0, *v1;
  SPK_TRY(ws_get(ctx, "vgk0", M * 8, (void **)&k0));
  SPK_TRY(ws_get(ctx, "vgk1", M * 8, (void **)&k1));
  SPK_TRY(ws_get(ctx, "vgv0", M * 8, (void **)&v0));
  SPK_TRY(ws_get(ctx, "vgv1", M * 8, (void **)&v1));
  const unsigned g = (unsigned)std::min<int64_t>(ceil_div(M, 256), 65536);
  hipLaunchKernelGGL(k_pair_keys, dim3(g), dim3(256), 0, ctx->stream, x, y, N,
                     k0, v0);
  SPK_TRY(check_launch("k_pair_keys"));
  size_t tmp_bytes = 0;
  SPK_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, k0, k1, v0,
                                             v1, (int)M, 0, 64, ctx->stream));
  void *tmp;
  SPK_TRY(ws_get(ctx, "vgtmp", tmp_bytes, &tmp));
  SPK_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, k0, k1, v0, v1,
                                             (int)M, 0, 64, ctx->stream));
  hipLaunchKernelGGL(k_pair_unpack, dim3(g), dim3(256), 0, ctx->stream, k1, v1,
                     M, pi, pj, pd);
  ctx->pairs_sorted = true;
  return check_launch("k_pair_unpack");
}

int spk_vgfit_evg_dev(spk_ctx *ctx, const int32_t *pi, const int32_t *pj,
                      const double *pd, int64_t M, int64_t N,
                      const double *vals, int64_t T, double mdr, int nk,
                      int classic, int max_bins, double *bin_h, double *bin_g,
                      int32_t *bin_n, int32_t *nbins) {
  if (!ctx || !pi || !pj || !pd || !vals || !bin_h || !bin_g || !bin_n ||
      !nbins)
    return set_error(SPK_EARG, "null argument");
  if (!(mdr > 0 && mdr <= 1)) return set_error(SPK_EARG, "mdr outside (0, 1]");
  if (nk <= 0) return set_error(SPK_EARG, "nk must be > 0");
  if (classic && nk > 64)
    return set_error(SPK_EARG, "the classic estimator supports nk <= 64");
  if (T <= 0) return SPK_OK;
  SPK_HIP(hipSetDevice(ctx->device));
  const int64_t S = std::min<int64_t>(T, 256);
  const int nch = (int)ceil_div(std::max<int64_t>(M, 1), kEvgChunk);
  // bins that a step can have, so that the grid covers every step's
  const int64_t nbm = std::min<int64_t>(max_bins, ceil_div(M, nk));
  int32_t *list;
  int64_t *cnt;
  SPK_TRY(ws_get(ctx, "vglist", S * M * 4, (void **)&list));
  SPK_TRY(ws_get(ctx, "vgcnt", S * (nch + 2) * 8, (void **)&cnt));
  int64_t *act = cnt + S * nch, *keep = act + S;
  for (int64_t t0 = 0; t0 < T; t0 += S) {
    const int Sb = (int)std::min<int64_t>(S, T - t0);
    const double *v = vals + t0 * N;
    if (nch <= kEvgSmall) {
      hipLaunchKernelGGL(k_evg_small, dim3(Sb), dim3(256), 0, ctx->stream, pi,
                         pj, pd, M, v, N, mdr, nk, classic, max_bins, list,
                         bin_h + t0 * max_bins, bin_g + t0 * max_bins,
                         bin_n + t0 * max_bins, nbins + t0);
      SPK_TRY(check_launch("k_evg"));
      continue;
    }
    hipLaunchKernelGGL(k_evg_count, dim3(nch, Sb), dim3(256), 0, ctx->stream,
                       pi, pj, M, v, N, cnt);
    hipLaunchKernelGGL(k_evg_scan, dim3(Sb), dim3(256), 0, ctx->stream, cnt,
                       nch, act);
    hipLaunchKernelGGL(k_evg_list, dim3(nch, Sb), dim3(256), 0, ctx->stream,
                       pi, pj, M, v, N, (const int64_t *)cnt, list);
    hipLaunchKernelGGL(k_evg_clip, dim3(Sb), dim3(64), 0, ctx->stream, pd, M,
                       mdr, nk, max_bins, (const int32_t *)list,
                       (const int64_t *)act, keep, nbins + t0);
    if (nbm > 0)
      hipLaunchKernelGGL(k_evg_bins, dim3((unsigned)ceil_div(nbm, 256), Sb),
                         dim3(256), 0, ctx->stream, pi, pj, pd, M, v, N, nk,
                         classic, max_bins, (const int32_t *)list,
                         (const int64_t *)keep, (const int32_t *)nbins + t0,
                         bin_h + t0 * max_bins, bin_g + t0 * max_bins,
                         bin_n + t0 * max_bins);
    SPK_TRY(check_launch("k_evg"));
  }
  return SPK_OK;
}

// Whether a caller is capturing the stream into a graph.
static bool stream_capturing(hipStream_t st) {
  if (!st) return false;  // the null stream cannot be captured
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cs) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return cs != hipStreamCaptureStatusNone;
}

// The evolution over the whole device (k_de_energy, k_de_step) in batches
// of at most kDeBatch (step, candidate) pairs, whose scratch is 162 KB
// (two components) to 213 KB (four) each.  The host reads the pairs still
// evolving every kDePoll generations (fits take 1 to 45).
constexpr int kDeBatch = 2048;
constexpr int kDePoll = 4;

static int de_device(spk_ctx *ctx, const double *bin_h, const double *bin_g,
                     const int32_t *nbins, int max_bins, const double *var,
                     int64_t T, const int32_t *dc, int n_cands, int maxiter,
                     int popmul, double tol, double range_ub, uint64_t seed,
                     const double *init, double spread, int pcap, int ds,
                     double *params, double *fun, int32_t *nit) {
  hipStream_t st = ctx->stream;
  const int64_t S =
      std::min<int64_t>(T, std::max<int64_t>(1, kDeBatch / n_cands));
  const int64_t nq = S * n_cands;
  double *pop, *trial, *energy, *part;
  unsigned long long *rngs;
  int32_t *done;
  SPK_TRY(ws_get(ctx, "vgde_pop", nq * pcap * ds * 8, (void **)&pop));
  SPK_TRY(ws_get(ctx, "vgde_trial", nq * pcap * ds * 8, (void **)&trial));
  SPK_TRY(ws_get(ctx, "vgde_energy", nq * pcap * 8, (void **)&energy));
  SPK_TRY(ws_get(ctx, "vgde_part", nq * kDeSplit * pcap * 8,
                 (void **)&part));
  SPK_TRY(ws_get(ctx, "vgde_rng", nq * 256 * 8, (void **)&rngs));
  SPK_TRY(ws_get(ctx, "vgde_done", 2 * nq * 4, (void **)&done));
  int32_t *list = done + nq;
  const size_t lds = (size_t)pcap * ds * sizeof(double);
  std::vector<int32_t> h_done(nq), h_list(nq);
  const unsigned gx =
      (unsigned)ceil_div(ceil_div(pcap, 64) * kDeSplit, 4);
  for (int64_t t0 = 0; t0 < T;) {
    // k_de's launches cover 65 535 steps and number them from zero
    const int64_t s0 = t0 % 65535;
    const int Sb =
        (int)std::min<int64_t>(std::min<int64_t>(S, T - t0), 65535 - s0);
    const double *h = bin_h + t0 * max_bins, *g = bin_g + t0 * max_bins;
    const int32_t *nbs = nbins + t0;
    const double *vr = var + t0;
    double *par = params + t0 * n_cands * kDeMaxD;
    double *fn = fun + t0 * n_cands;
    int32_t *ni = nit + t0 * n_cands;
    hipLaunchKernelGGL(k_de_init, dim3(n_cands, Sb), dim3(256), 0, st, h, g,
                       nbs, max_bins, vr, dc, n_cands, popmul, range_ub,
                       (unsigned long long)seed, (int)s0,
                       init ? init + t0 * n_cands * kDeMaxD : nullptr, spread,
                       pcap, ds, pop, rngs, done, fn, ni);
    int na = Sb * n_cands;
    const int32_t *lst = nullptr;
    auto generation = [&](int it) {
      hipLaunchKernelGGL(k_de_energy, dim3(gx, na), dim3(256), 0, st, h, g,
                         nbs, max_bins, vr, dc, n_cands, popmul, range_ub,
                         pcap, ds, (const double *)(it ? trial : pop), lst,
                         (const int32_t *)done, part);
      hipLaunchKernelGGL(k_de_step, dim3(na), dim3(256), lds, st, h, g, nbs,
                         max_bins, vr, dc, n_cands, it, maxiter, popmul, tol,
                         range_ub, pcap, ds, pop, trial, energy,
                         (const double *)part, rngs, lst, done, par, fn, ni);
    };
    generation(0);
    for (int it = 1; it <= maxiter && na > 0; ++it) {
      generation(it);
      if (it % kDePoll && it < maxiter) continue;
      SPK_TRY(check_launch("k_de_step"));
      SPK_TRY(d2h(ctx, h_done.data(), done, (size_t)Sb * n_cands * 4));
      na = 0;
      for (int k = 0; k < Sb * n_cands; ++k)
        if (!h_done[k]) h_list[na++] = k;
      if (na > 0) SPK_TRY(h2d(ctx, list, h_list.data(), (size_t)na * 4));
      lst = list;
    }
    SPK_TRY(check_launch("k_de_energy"));
    t0 += Sb;
  }
  return SPK_OK;
}

static int de_launch(spk_ctx *ctx, const double *bin_h, const double *bin_g,
                     const int32_t *nbins, int max_bins, const double *var,
                     int64_t T, const int32_t *cands, int n_cands, int maxiter,
                     int popmul, double tol, double range_ub, uint64_t seed,
                     const double *init, double spread, double *params,
                     double *fun, int32_t *nit) {
  if (!ctx || !bin_h || !bin_g || !nbins || !var || !cands || !params ||
      !fun || !nit)
    return set_error(SPK_EARG, "null argument");
  if (n_cands <= 0 || n_cands > 64) return set_error(SPK_EARG, "bad n_cands");
  if (popmul <= 0 || maxiter <= 0) return set_error(SPK_EARG, "bad DE sizes");
  for (int c = 0; c < n_cands; ++c)
    if (cands[c * 6] < 1 || cands[c * 6] > 4)
      return set_error(SPK_EARG, "candidate %d: 1..4 components", c);
  if (init && !(spread >= 0.0 && spread <= 20.0))
    return set_error(SPK_EARG, "spread outside [0, 20]");
  if (T <= 0) return SPK_OK;
  SPK_HIP(hipSetDevice(ctx->device));
  int32_t *dc;
  SPK_TRY(ws_get(ctx, "vgcand", n_cands * 6 * 4, (void **)&dc));
  SPK_TRY(h2d(ctx, dc, cands, n_cands * 6 * 4));
  // LDS rows of the largest candidate: stride ds parameters, pcap members
  int ds = 0, pcap = 0;
  for (int c = 0; c < n_cands; ++c) {
    const int D = 2 * cands[c * 6];
    ds = std::max(ds, D);
    pcap = std::max(pcap, de_pop(popmul, D));
  }
  // Few bins: one workgroup per (step, candidate) evolves it by itself.  A
  // generation then takes 5 us and, per bin, component and 256 members, 0.05 us
  // (eight times that for pow and sin); over the whole device it takes 20 to
  // 50 us for its launches and the host's look, and 0.03 to 0.1 us per pair.
  // The line is the best fit to 184 calls of 1 to 600 bins and 2 to 22 000
  // pairs.  One step x 7 candidates of Sph, Exp and Gau, ms by the one and the
  // other: 12 stations (1 bin) 1.1 and 5.4, 60 (21 bins) 0.90 and 1.31, 130
  // (120 bins) 2.4 and 1.7; 200 steps: 2.6 and 17, 2.0 and 4.4, 5.2 and 6.2.
  // Both give the same bits.  Captured launches cannot be followed by host
  // reads and take the first form.
  const size_t lds = de_lds_bytes(pcap, ds);
  const int64_t pairs = T * n_cands;
  int64_t work = 0;  // of the slowest candidate, per bin
  for (int c = 0; c < n_cands; ++c) {
    const int32_t *cd = cands + c * 6;
    int64_t w = 0;
    for (int k = 0; k < cd[0]; ++k)
      w += cd[1 + k] == SPK_VG_POW || cd[1 + k] == SPK_VG_HOL ? 8 : 1;
    work = std::max(work, w * ceil_div(de_pop(popmul, 2 * cd[0]), 256));
  }
  auto few = [&](int64_t nb) { return nb * work <= 500 + pairs / 3; };
  if (!stream_capturing(ctx->stream) && !few(max_bins)) {
    std::vector<int32_t> h_nb(T);
    SPK_TRY(d2h(ctx, h_nb.data(), nbins, (size_t)T * 4));
    if (!few(*std::max_element(h_nb.begin(), h_nb.end()))) {
      const int rc = de_device(ctx, bin_h, bin_g, nbins, max_bins, var, T, dc,
                               n_cands, maxiter, popmul, tol, range_ub, seed,
                               init, spread, pcap, ds, params, fun, nit);
      // without the memory for its populations, the form that needs none
      if (rc != SPK_ENOMEM) return rc;
      (void)hipGetLastError();
    }
  }
  if (lds > 64 * 1024)
    SPK_HIP(hipFuncSetAttribute((const void *)k_de,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  for (int64_t t0 = 0; t0 < T; t0 += 65535) {
    const int Tb = (int)std::min<int64_t>(65535, T - t0);
    hipLaunchKernelGGL(k_de, dim3(n_cands, Tb), dim3(256), lds, ctx->stream,
                       bin_h + t0 * max_bins, bin_g + t0 * max_bins,
                       nbins + t0, max_bins, var + t0, dc, n_cands, maxiter,
                       popmul, tol, range_ub, (unsigned long long)seed,
                       init ? init + t0 * n_cands * kDeMaxD : nullptr, spread,
                       pcap, ds, params + t0 * n_cands * kDeMaxD,
                       fun + t0 * n_cands,
                       nit + t0 * n_cands);
    SPK_TRY(check_launch("k_de"));
  }
  return SPK_OK;
}

int spk_vgfit_de_dev(spk_ctx *ctx, const double *bin_h, const double *bin_g,
                     const int32_t *nbins, int max_bins, const double *var,
                     int64_t T, const int32_t *cands, int n_cands, int maxiter,
                     int popmul, double tol, double range_ub, uint64_t seed,
                     double *params, double *fun, int32_t *nit) {
  return de_launch(ctx, bin_h, bin_g, nbins, max_bins, var, T, cands, n_cands,
                   maxiter, popmul, tol, range_ub, seed, nullptr, 0.0, params,
                   fun, nit);
}

int spk_vgfit_de_seeded_dev(spk_ctx *ctx, const double *bin_h,
                            const double *bin_g, const int32_t *nbins,
                            int max_bins, const double *var, int64_t T,
                            const int32_t *cands, int n_cands, int maxiter,
                            int popmul, double tol, double range_ub,
                            uint64_t seed, const double *init, double spread,
                            double *params, double *fun, int32_t *nit) {
  if (!init) return set_error(SPK_EARG, "null argument");
  return de_launch(ctx, bin_h, bin_g, nbins, max_bins, var, T, cands, n_cands,
                   maxiter, popmul, tol, range_ub, seed, init, spread, params,
                   fun, nit);
}

}  // extern "C"
