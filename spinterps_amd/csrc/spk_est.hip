// Dual-form estimates of the batched path where no variance is wanted
// (SPK_M_SK, SPK_M_EDK, SPK_M_OK without its variance): per step and cell
//     est = k.alpha + f.h,  k_i = c0 - gamma(d_i) (OK / EDK) or the covariance
// sum (SK), interp/steps.py:403-435 in the dual form of spk_factor.hip.
#include "spk_krige.h"

namespace spk {

// grid (ceil(rec_stride(N) / 256), steps)
__global__ __launch_bounds__(256) void k_stn_rec(
    const double *__restrict__ sx, const double *__restrict__ sy,
    const int32_t *__restrict__ idx, int64_t N, const StepSc *__restrict__ sc,
    const double *__restrict__ V, int64_t ldv, int64_t ld,
    StnRec *__restrict__ rec) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int j = blockIdx.x * 256 + threadIdx.x;
  const int n = sc[s].n;
  if (j >= (n + 15) / 16 * 16) return;
  StnRec r = {kFarCoord, kFarCoord, 0.0, 0.0, 0.0, {0.0, 0.0, 0.0}};
  if (j < n) {
    const int g = idx[(int64_t)s * N + j];
    const double *v = V + (int64_t)s * ldv + j;  // alpha, w, dalpha: ld apart
    r.x = coord_stn(sx[g]);
    r.y = coord_stn(sy[g]);
    r.alpha = v[0];
    r.w = v[ld];
    r.dalpha = v[2 * ld];
  }
  rec[s * rec_stride(N) + j] = r;
}

int stn_records(hipStream_t st, const double *sx, const double *sy,
                const int32_t *idx, int64_t N, const StepSc *sc,
                const double *V, int64_t ldv, int64_t ld, int S, StnRec *rec) {
  hipLaunchKernelGGL(k_stn_rec, dim3((unsigned)ceil_div(rec_stride(N), 256), S),
                     dim3(256), 0, st, sx, sy, idx, N, sc, V, ldv, ld, rec);
  return check_launch("k_stn_rec");
}

// Sums of one cell over stations [j0, j1) of a step: k.alpha, k.w (SKW only)
// and k.dalpha.  cov(dx, dy) is k.  The records' addresses are uniform, so
// their fields arrive as scalar operands.
template <bool SKW, typename F>
__device__ inline void est_sum(const StnRec *__restrict__ rec, int j0, int j1,
                               double x, double y, double &e, double &a,
                               double &ke, F cov) {
#pragma unroll 4
  for (int j = j0; j < j1; ++j) {
    const double k = cov(x - rec[j].x, y - rec[j].y);
    e = fma(k, rec[j].alpha, e);
    if (SKW) a = fma(k, rec[j].w, a);
    ke = fma(k, rec[j].dalpha, ke);
  }
}

// One cell per thread, all stations of the step; grid (cells / 256, steps).
// A single bounded model with or without a nugget is evaluated as
// k = off + s f(h) with off = c0 - nug - s (0 for the usual c0, and for SK),
// f = 2^(c h), 2^(c h^2) or 1 - 1.5 u + 0.5 u^3, u = min(h / r, 1): 27, 18
// and 17 FP64 instructions per station and cell with the sums, no branch and
// no LDS.  Bound by FP64 VALU issue.  Other variograms (several components,
// unbounded models, a positive min_vg_val, which can cut small values) go
// through the general evaluation.  For systems of 900 stations, 250 000 cells
// and 32 steps the earlier kernel, which staged five fields per station in
// LDS, looked for the nearest station and looped over components with
// library sqrt and exp, took 23 ms.
template <bool GEN, bool SKW>
__global__ __launch_bounds__(256) void k_est(
    const double *__restrict__ sx, const double *__restrict__ sy,
    const int32_t *__restrict__ idx, int64_t N,
    const StnRec *__restrict__ recs, const double *__restrict__ zact,
    int64_t ldz, StepSc *__restrict__ sc, const spk_vg *__restrict__ vgs,
    const double *__restrict__ cx, const double *__restrict__ cy, int64_t Cs,
    int64_t C, const double *__restrict__ cell_drift,
    const int32_t *__restrict__ perm, int method, int m, int skm,
    double min_vg_val, double *__restrict__ est, int64_t ldo) {
  const int sl = blockIdx.y;
  const StepSc *stp = sc + sl;
  if (stp->status) return;
  const int n = stp->n;
  const int tid = threadIdx.x;
  __shared__ VgFast vf;
  if (tid == 0) vg_fast_init(vgs[sl], vf);
  __syncthreads();
  const int64_t c = blockIdx.x * (int64_t)256 + tid;
  const bool valid = c < Cs;
  const double xr = valid ? cx[c] : 0.0, yr = valid ? cy[c] : 0.0;
  const bool bounded = vg_bounded(vgs[sl]);
  const double x = bounded ? coord_fast(xr) : xr;
  const double y = bounded ? coord_fast(yr) : yr;
  const StnRec *rec = recs + sl * rec_stride(N);
  const bool sk = method == SPK_M_SK;
  const double c0 = stp->c0;
  VgOne o;
  int one = vg_one_of(vf, o);
  // entries <= min_vg_val become zero (pyx:217): with min_vg_val <= 0 and
  // nonnegative sills that changes nothing
  if (!(min_vg_val <= 0.0 && o.s >= 0.0 && o.nug >= 0.0)) one = -1;
  double e = 0.0, a = 0.0, ke = 0.0;
  const double s = o.s, off = sk ? 0.0 : c0 - o.nug - o.s;
  if (one == SPK_VG_EXP) {
    const double q = o.c1;
    est_sum<SKW>(rec, 0, n, x, y, e, a, ke, [&](double dx, double dy) {
      return fma(s, exp2_neg(dist_fast(dx, dy) * q), off);
    });
  } else if (one == SPK_VG_GAU) {
    const double q = o.c1;
    est_sum<SKW>(rec, 0, n, x, y, e, a, ke, [&](double dx, double dy) {
      return fma(s, exp2_neg(fma(dx, dx, dy * dy) * q), off);
    });
  } else if (one == SPK_VG_SPH) {
    const double q = 1.0 / o.r, top = off + s;
    est_sum<SKW>(rec, 0, n, x, y, e, a, ke, [&](double dx, double dy) {
      const double h = dist_fast(dx, dy) * q;
      const double u = h < 1.0 ? h : h >= 1.0 ? 1.0 : h;  // NaN stays NaN
      return fma(s * u, fma(u * u, 0.5, -1.5), top);
    });
  } else {
    // the evaluation of the variance path's kernel (spk_cells.hip)
    const bool simp = !GEN || vg_simple(vgs[sl]);
    est_sum<SKW>(rec, 0, n, x, y, e, a, ke, [&](double dx, double dy) {
      const double h = simp ? dist_fast(dx, dy) : dist2(dx, dy, 0.0, 0.0);
      const double g =
          GEN ? vg_fast_entry(vf, h, sk ? 1 : 0, min_vg_val)
              : vg_simple_entry(vf, h, sk ? 1 : 0, min_vg_val);
      return sk ? g : c0 - g;
    });
  }
  // the reference's SK takes the nearest station where the weights do not
  // sum to about one (interp/steps.py:418-427)
  const double *z = zact + (int64_t)sl * ldz;
  const bool far = SKW && valid && !skm && !isclose1(a);
  int bi = 0;
  if (SKW && __syncthreads_or(far ? 1 : 0)) {
    __shared__ double2 st[256];
    __shared__ int id[256];
    const int32_t *my = idx + (int64_t)sl * N;
    double best = INFINITY;
    int bid = 0;
    for (int base = 0; base < n; base += 256) {
      __syncthreads();
      if (base + tid < n) {
        id[tid] = my[base + tid];
        st[tid] = double2{sx[id[tid]], sy[id[tid]]};
      }
      __syncthreads();
      const int cnt = min(256, n - base);
      for (int j = 0; j < cnt; ++j) {
        const double d = dist2(xr, yr, st[j].x, st[j].y);
        // ties go to the lower station index, whatever order the step's
        // stations are compacted in
        if (d < best || (d == best && id[j] < bid)) {
          best = d;
          bi = base + j;
          bid = id[j];
        }
      }
    }
  }
  if (!valid) return;
  const int64_t oc = perm ? (int64_t)perm[c] : c;
  // residual check: the change by the second refinement step (kRefineTol)
  double de = ke, ev;
  if (method == SPK_M_OK) {
    ev = e + stp->a0;
    de += stp->dh[0];
  } else if (method == SPK_M_EDK) {
    ev = e + stp->h[0];
    de += stp->dh[0];
    for (int k = 0; k < m; ++k) {
      const double f = cell_drift[(int64_t)k * C + oc];
      ev += stp->h[1 + k] * f;
      de += stp->dh[1 + k] * f;
    }
  } else if (skm) {
    // SK with the step mean m as known mean: m + k^T C^-1 (z - m 1)
    // = k.alpha + m (1 - k.w)
    ev = e + stp->mean * (1.0 - a);
  } else {  // the reference's SK
    ev = far ? z[bi] : e;
  }
  const bool ill = fabs(de) > kRefineTol * fmax(fabs(ev), 1e-3 * stp->zabs);
  if (ill && !(stp->flags & SPK_ST_ILLCOND))
    atomicOr(&sc[sl].flags, SPK_ST_ILLCOND);
  est[(int64_t)sl * ldo + oc] = ev;
}

int est_steps(hipStream_t st, const double *sx, const double *sy,
              const int32_t *idx, int64_t N, const StnRec *rec,
              const double *zact, int64_t ldz, StepSc *sc, const spk_vg *vgs,
              int S, bool simple, const double *cx, const double *cy,
              int64_t Cs, int64_t C, const double *cell_drift,
              const int32_t *perm, int method, int m, int skm,
              double min_vg_val, double *est, int64_t ldo) {
  const bool skw = method == SPK_M_SK;
  auto k = simple ? (skw ? k_est<false, true> : k_est<false, false>)
                  : (skw ? k_est<true, true> : k_est<true, false>);
  hipLaunchKernelGGL(k, dim3((unsigned)ceil_div(Cs, 256), S), dim3(256), 0, st,
                     sx, sy, idx, N, rec, zact, ldz, sc, vgs, cx, cy, Cs, C,
                     cell_drift, perm, method, m, skm, min_vg_val, est, ldo);
  return check_launch("k_est");
}

}  // namespace spk
