// IDW as a masked contraction on FP64 MFMA (interp/steps.py:293-313,
// pyx:784-808).
//
// The reference, per cell of a time group: d <- d / max(d), w_i = 1 / d_i^p
// over the group's active stations, then per step sum(w z) / sum(w).  The
// factor max(d)^p is common to numerator and denominator, so with
// W[c, i] = d_ci^-p over all N stations and the step's mask M[t, i] (1 where
// station i has a value) the fields are
//     num = (Z . M) W^T,   den = M W^T,   est[t, c] = num[t, c] / den[t, c],
// two GEMMs over the stations that share W, which is generated on the fly
// (once per block and chunk of stations, used for BS steps x 2 sums).  The
// results differ from the reference's by rounding only (the sums run in
// another order, without the normalisation).
//
// Orientation: the MFMA output rows are steps and its columns cells, so the
// numerator and denominator of one (step, cell) land in the same lane and
// register of two accumulator tiles.  Block tile BS steps x 32 NW cells, a
// wave BS steps x 32 cells (BS / 16 x 2 tiles of 16 x 16, for each of num and
// den), stations in chunks of 16 through two LDS buffers, one barrier per
// chunk: the next chunk's weights and values are formed before the current
// one is multiplied, by the other blocks' waves meanwhile.
//
// Bound: FP64 MFMA issue (77 TF with registers only; 64 cycles for 16 x 16 x
// 4), and the FP64 VALU work between, which shares its units: per wave and
// chunk 64 products (4 096 cycles) and, for p = 2, some 180 vector
// instructions, hence the reciprocal by hand, stations padded by repetition
// and the zero-distance test by ballot (250 before).  365 steps x 1 000
// stations x 250 000 cells: 6.9 ms, 53 TF; with 32 steps per block, a
// division per weight, station loads next to it and three barriers per
// chunk 9.1 ms.  One step x 100 stations x 2 500 cells: 13 us for 24.
//
// A cell at zero distance from a station has an infinite weight: the
// reference then returns NaN for the steps where that station has a value.
// Such cells (rare) are recomputed per step in the reference's arithmetic.
#include "spk_krige.h"

namespace spk {

typedef double idw_d4 __attribute__((ext_vector_type(4)));

__device__ inline idw_d4 idw_mfma(double a, double b, idw_d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// One (cell, step) in the reference's arithmetic: w = 1 / (d / dmax)^p over
// the step's active stations (pyx:784-808), sum(w z) / sum(w).
__device__ double idw_cell_ref(double x, double y, const double *sx,
                               const double *sy, const int32_t *my,
                               const double *z, int n, double p, int *bad) {
#pragma clang fp contract(off)
  double dmax = 0.0;
  for (int j = 0; j < n; ++j) dmax = fmax(dmax, dist2(x, y, sx[my[j]], sy[my[j]]));
  double ws = 0.0, wz = 0.0;
  for (int j = 0; j < n; ++j) {
    double d = dist2(x, y, sx[my[j]], sy[my[j]]);
    if (dmax > 0) d = d / dmax;
    const double wj = 1.0 / (p == 2.0 ? d * d : pow(d, p));
    ws = ws + wj;
    wz = wz + wj * z[j];
  }
  if (!(ws >= 1e-14)) *bad = 1;  // interp/steps.py:305
  return wz / ws;
}

// s2^(-p / 2) for s2 > 0.  KIND 0: p = 2; 1: p a multiple of 1/2 up to 8,
// by squaring from 1 / d (p2 = 2 p, within p ulp; a pow() per weight costs
// some 150 FP64 instructions, as much as half a chunk's products); 2: others.
template <int KIND>
__device__ inline double idw_weight(double s2, double p, int p2) {
  if constexpr (KIND == 0) {
    // the hardware's reciprocal (5e-8), one step of third order; half the
    // instructions of a division
    const double y = __builtin_amdgcn_rcp(s2);
    const double e = fma(-s2, y, 1.0);
    return __builtin_amdgcn_div_fixup(fma(y, fma(e, e, e), y), s2, 1.0);
  }
  if constexpr (KIND == 2) return 1.0 / pow(sqrt(s2), p);
  double q = 1.0 / sqrt(s2);
  double w = p2 & 1 ? sqrt(q) : 1.0;
  for (int e = p2 >> 1; e; e >>= 1) {
    if (e & 1) w *= q;
    q *= q;
  }
  return w;
}

// grid (ceil(C / (32 NW)), ceil(S / BS)), 64 NW threads; vals [S x N] the
// launch's steps (NaN = no value), sc [S] their records (k_compact), est
// [S x C]; info and kappa (may be null) [S] are the steps' status words and
// condition estimates.  Special steps (one station, mean fill) are filled here too; a
// step without stations is left alone (interp/steps.py:280-283, 325-331).
template <int BS, int NW, int KIND>
__global__ __launch_bounds__(64 * NW, 2) void k_idw_mfma(
    const double *__restrict__ sx, const double *__restrict__ sy, int64_t N,
    const double *__restrict__ vals, int S, const StepSc *__restrict__ sc,
    const int32_t *__restrict__ idx, const double *__restrict__ zact,
    int64_t ldz, const double *__restrict__ cx, const double *__restrict__ cy,
    int64_t C, double p, int p2, double *__restrict__ est,
    int *__restrict__ bad, int32_t *__restrict__ info,
    double *__restrict__ kappa) {
  constexpr int NT = 64 * NW, BC = 32 * NW, KC = 16, TS = BS / 16;
  constexpr int AL = BS * KC / NT;          // values per thread and chunk
  __shared__ double Ws[2][KC][BC + 16];     // W[station][cell]
  __shared__ double As[2][2][BS][KC + 2];   // z . m and m, [step][station]
  __shared__ double Ps[2][2][KC];           // x and y of the stations
  __shared__ int coinc[BC];                 // cell at a station
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int64_t c0 = blockIdx.x * (int64_t)BC;
  const int t0 = blockIdx.y * BS;
  // the thread's cell and first station of a chunk for the W tile
  const int wc = tid % BC, wk = tid / BC;
  const int64_t gc = c0 + wc;
  const bool have = gc < C;
  const double x = have ? cx[gc] : 0.0, y = have ? cy[gc] : 0.0;
  if (tid < BC) coinc[tid] = 0;
  if (blockIdx.x == 0)
    for (int u = tid; u < BS && t0 + u < S; u += NT) {
      info[t0 + u] = sc[t0 + u].status | sc[t0 + u].flags;
      if (kappa) kappa[t0 + u] = sc[t0 + u].kappa;
    }
  idw_d4 acc[2][TS][2];  // [num/den][step tile][cell tile]
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int a = 0; a < TS; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[q][a][b] = idw_d4{0, 0, 0, 0};
  // values and stations of a chunk (beyond the last station its position
  // again and no value): read two chunks ahead, so that no wait
  // for memory stands between two chunks' products (with the stations read
  // where the weights are formed, the matrix cores were busy 62 % of the time)
  double va[AL], pa = 0.0;
  unsigned long long hits = 0;  // the wave's lanes with a cell at a station
  const double *ps = tid & KC ? sy : sx;
  auto fetch_stn = [&](int64_t k0) {
    const int64_t i = k0 + (tid & (KC - 1));
    if (tid < 2 * KC) pa = ps[i < N ? i : N - 1];
  };
  auto put_stn = [&](int buf) {
    if (tid < 2 * KC) Ps[buf][tid / KC][tid % KC] = pa;
  };
  const double *pv[AL];
#pragma unroll
  for (int u = 0; u < AL; ++u)
    pv[u] = vals + (int64_t)min(t0 + (tid + NT * u) / KC, S - 1) * N +
            (tid & (KC - 1));
  auto fetch = [&](int64_t k0) {
#pragma unroll
    for (int u = 0; u < AL; ++u) {
      const int64_t i = k0 + (tid & (KC - 1));
      va[u] = i < N ? pv[u][k0] : NAN;
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int u = 0; u < AL; ++u) {
      const int e = tid + NT * u;
      const bool has = !isnan(va[u]);
      As[buf][0][e >> 4][e & 15] = has ? va[u] : 0.0;
      As[buf][1][e >> 4][e & 15] = has ? 1.0 : 0.0;
    }
#pragma unroll(KIND == 2 ? 1 : KC / 2)
    for (int u = 0; u < KC / 2; ++u) {
      const int k = wk + 2 * u;
      double s2;
      {
#pragma clang fp contract(off)
        const double dx = x - Ps[buf][0][k], dy = y - Ps[buf][1][k];
        s2 = (dx * dx) + (dy * dy);
      }
      // a cell at a station has an infinite weight: epilogue
      const bool pos = s2 > 0.0;
      const double v = idw_weight<KIND>(s2, p, p2);
      const double w = pos ? v : 0.0;
      hits |= __ballot(!pos);
      Ws[buf][k][wc] = w;
    }
  };
  fetch_stn(0);
  put_stn(0);
  fetch(0);
  fetch_stn(KC);
  __syncthreads();
  put(0);
  put_stn(1);
  fetch(KC);
  fetch_stn(2 * KC);
  __syncthreads();
  int buf = 0;
  for (int64_t k0 = 0; k0 < N; k0 += KC, buf ^= 1) {
    // stations of chunk c are in Ps[c & 1] from the end of iteration c - 2
    if (k0 + KC < N) {
      put(buf ^ 1);
      put_stn(buf);
      fetch(k0 + 2 * KC);
      fetch_stn(k0 + 3 * KC);
    }
#pragma unroll
    for (int kk = 0; kk < KC / 4; ++kk) {
      const int k = kk * 4 + lg;
      double bf[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) bf[b] = Ws[buf][k][wave * 32 + b * 16 + li];
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int a = 0; a < TS; ++a) {
          const double af = As[buf][q][a * 16 + li][k];
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[q][a][b] = idw_mfma(af, bf[b], acc[q][a][b]);
        }
    }
    __syncthreads();
  }
  if ((hits >> lane & 1) && have) coinc[wc] = 1;
  __syncthreads();
  // epilogue: lane (lg, li) holds rows lg + 4 r of each tile, column li
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int cl = wave * 32 + b * 16 + li;
    const int64_t c = c0 + cl;
    if (c >= C || coinc[cl]) continue;
#pragma unroll
    for (int a = 0; a < TS; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = t0 + a * 16 + lg + 4 * r;
        if (t >= S) continue;
        const int status = sc[t].status;
        double e;
        if (status == SPK_ST_NOSTNS) continue;
        if (status == SPK_ST_ONESTN) {
          e = zact[(int64_t)t * ldz];
        } else if (status == SPK_ST_MEANFILL) {
          e = sc[t].mean;
        } else {
          const double num = acc[0][a][b][r], den = acc[1][a][b][r];
          // the reference's check on the normalised weight sum (at least
          // one, when finite) fails only for a non-finite or zero sum
          if (!(den > 0.0) || !isfinite(den)) *bad = 1;
          e = num / den;
        }
        est[(int64_t)t * C + c] = e;
      }
  }
  // the cells at a station, if any
  for (int e = tid; e < BC * BS; e += NT) {
    const int cl = e % BC, t = t0 + e / BC;
    if (!coinc[cl] || t >= S) continue;
    const StepSc &q = sc[t];
    const double *z = zact + (int64_t)t * ldz;
    double v;
    if (q.status == SPK_ST_NOSTNS) continue;
    if (q.status == SPK_ST_ONESTN)
      v = z[0];
    else if (q.status == SPK_ST_MEANFILL)
      v = q.mean;
    else
      v = idw_cell_ref(cx[c0 + cl], cy[c0 + cl], sx, sy, idx + (int64_t)t * N,
                       z, q.n, p, bad);
    est[(int64_t)t * C + c0 + cl] = v;
  }
}

// Steps per block: the more, the fewer times a weight is formed, but absent
// steps of a block cost as much as others and the grid has to fill the device
// (two blocks of four waves per CU): the largest of 64, 48, 32 and 16 that
// does both, one wave per block of 16 steps where none does.  The steps beyond
// whole blocks of 64 go by themselves, unless all steps together leave the
// device idle: then a second launch only adds its latency (70 steps x 300
// stations x 1 000 cells, p = 2.3: 246 us, in one launch 148).
template <int BS, int NW>
static void idw_launch(hipStream_t st, const double *sx, const double *sy,
                       int64_t N, const double *vals, int S, const StepSc *sc,
                       const int32_t *idx, const double *zact, int64_t ldz,
                       const double *cx, const double *cy, int64_t C, double p,
                       double *est, int *bad, int32_t *info, double *kappa) {
  const double pp = 2.0 * p;
  const int p2 = pp >= 1.0 && pp <= 16.0 && pp == floor(pp) ? (int)pp : 0;
  auto k = p2 == 4 ? k_idw_mfma<BS, NW, 0>
                   : p2 ? k_idw_mfma<BS, NW, 1> : k_idw_mfma<BS, NW, 2>;
  hipLaunchKernelGGL(k, dim3((unsigned)ceil_div(C, 32 * NW),
                             (unsigned)ceil_div(S, BS)),
                     dim3(64 * NW), 0, st, sx, sy, N, vals, S, sc, idx, zact,
                     ldz, cx, cy, C, p, p2, est, bad, info, kappa);
}

int idw_steps(hipStream_t st, const double *sx, const double *sy, int64_t N,
              const double *vals, int S, const StepSc *sc, const int32_t *idx,
              const double *zact, int64_t ldz, const double *cx,
              const double *cy, int64_t C, double p, double *est, int *bad,
              int32_t *info, double *kappa) {
  auto go = [&](int t0, int n) {
    const int64_t ct = ceil_div(C, 128);
    auto l = ct * ceil_div(n, 64) >= 512 && n > 48
                 ? idw_launch<64, 4>
                 : ct * ceil_div(n, 48) >= 512 && n > 32
                 ? idw_launch<48, 4>
                 : ct * ceil_div(n, 32) >= 512 && n > 16
                       ? idw_launch<32, 4>
                       : ct * ceil_div(n, 16) >= 512 ? idw_launch<16, 4>
                                                     : idw_launch<16, 1>;
    l(st, sx, sy, N, vals + t0 * N, n, sc + t0, idx + t0 * N, zact + t0 * ldz,
      ldz, cx, cy, C, p, est + t0 * C, bad, info + t0,
      kappa ? kappa + t0 : nullptr);
  };
  const int full =
      ceil_div(C, 128) * ceil_div(S, 16) < 512 ? 0 : S / 64 * 64;
  if (full > 0) go(0, full);
  if (S > full) go(full, S - full);
  return check_launch("k_idw_mfma");
}

}  // namespace spk
