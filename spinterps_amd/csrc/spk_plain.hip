// Cell kernels of the plain FP64 path (SPK_P_FP64) and of the contraction
// of pseudo-inverse steps: per cell lambda = K^-1 rhs (interp/steps.py:
// 403-434) for every step of a launch.
//
//  k_plain_rhs   the right-hand sides R [(n + p) x cells] of every step
//                (interp/steps.py:203-234)
//  k_plain_gemm  lambda = M R by FP64 MFMA over (64 rows, 128 cells) tiles,
//                reduced at once to each tile's share of lambda.z, sum
//                lambda and lambda.gamma + 2 mu per cell
//  k_plain_fin   the shares summed over the row tiles, the reference's
//                sum-of-weights test with its nearest-station fallback, the
//                outputs and the residual flag
#include "spk_krige.h"

namespace spk {

typedef double p4_t __attribute__((ext_vector_type(4)));

// One column of a station chunk: value of every station of the chunk at
// the thread's cell, stored row by row.
template <typename F>
__device__ inline void plain_col(const double2 *st, int cnt, double x,
                                 double y, double *R, int64_t ldr, F val) {
#pragma unroll 4
  for (int j = 0; j < cnt; ++j)
    R[(int64_t)j * ldr] = val(dist_fast(x - st[j].x, y - st[j].y));
}

// grid (cells / 256, stations / 128, steps).  One bounded model with or
// without a nugget runs through vg_one's loop (constants folded, no
// component switch inside), other variograms through vg_entry.  The
// stations are split over blocks so that a small grid of cells still fills
// the device: 24 steps of 100 stations and 2 500 cells took one launch of
// ten blocks per step, 66 us each; all steps at once take 17 us.  Large
// calls are bound by the writes of R (900 stations x 250 000 cells: 1.7 ms
// per step with one thread per cell walking all stations through the
// component loop, 0.34 ms now, 5.2 TB/s).
__global__ __launch_bounds__(256) void k_plain_rhs(
    const double *__restrict__ sx, const double *__restrict__ sy,
    const int32_t *__restrict__ idx, int64_t N, const StepSc *__restrict__ sc,
    const spk_vg *__restrict__ vgs, const double *__restrict__ cx,
    const double *__restrict__ cy, int64_t Cs, int64_t ldd,
    const double *__restrict__ cell_drift, int method, int m,
    double min_vg_val, double *__restrict__ R, int64_t ldr, int64_t strideR,
    const int *__restrict__ ccount) {
  const int s = blockIdx.z;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int j0 = blockIdx.y * kPlainStn;
  if (ccount) Cs = min(Cs, (int64_t)*ccount);
  if (j0 >= n || blockIdx.x * (int64_t)256 >= Cs) return;
  __shared__ double2 st[kPlainStn];
  __shared__ spk_vg vg;
  __shared__ VgOne one;
  __shared__ int model;
  const int tid = threadIdx.x;
  const int covar = method == SPK_M_SK ? 1 : 0;
  const int32_t *my = idx + (int64_t)s * N + j0;
  if (tid < kPlainStn && j0 + tid < n) {
    const int g = my[tid];
    st[tid] = double2{coord_stn(sx[g]), coord_stn(sy[g])};
  }
  if (tid == kPlainStn) {
    vg = vgs[s];
    VgFast f;
    vg_fast_init(vg, f);
    VgOne o;
    model = vg_one_of(f, o);
    one = o;
  }
  __syncthreads();
  const int64_t c = blockIdx.x * (int64_t)256 + tid;
  if (c >= Cs) return;
  const int cnt = min(kPlainStn, n - j0);
  const double x = coord_fast(cx[c]), y = coord_fast(cy[c]);
  double *Rs = R + (int64_t)s * strideR;
  double *Rc = Rs + (int64_t)j0 * ldr + c;
  const VgOne o = one;
  // covariance form: sill - gamma of the model (the nugget's is zero)
  const double sill = o.s;
  VgOne oz = o;
  oz.nug = 0.0;
  auto cov = [&](double g) {
    const double w = sill - g;
    return w <= min_vg_val ? 0.0 : w;
  };
  if (model == SPK_VG_SPH) {
    if (covar)
      plain_col(st, cnt, x, y, Rc, ldr, [&](double h) {
        return cov(vg_one<SPK_VG_SPH>(oz, h, -INFINITY));
      });
    else
      plain_col(st, cnt, x, y, Rc, ldr, [&](double h) {
        return vg_one<SPK_VG_SPH>(o, h, min_vg_val);
      });
  } else if (model == SPK_VG_EXP) {
    if (covar)
      plain_col(st, cnt, x, y, Rc, ldr, [&](double h) {
        return cov(vg_one<SPK_VG_EXP>(oz, h, -INFINITY));
      });
    else
      plain_col(st, cnt, x, y, Rc, ldr, [&](double h) {
        return vg_one<SPK_VG_EXP>(o, h, min_vg_val);
      });
  } else if (model == SPK_VG_GAU) {
    if (covar)
      plain_col(st, cnt, x, y, Rc, ldr, [&](double h) {
        return cov(vg_one<SPK_VG_GAU>(oz, h, -INFINITY));
      });
    else
      plain_col(st, cnt, x, y, Rc, ldr, [&](double h) {
        return vg_one<SPK_VG_GAU>(o, h, min_vg_val);
      });
  } else {
    for (int j = 0; j < cnt; ++j)
      Rc[(int64_t)j * ldr] =
          vg_entry(vg, dist2(cx[c], cy[c], sx[my[j]], sy[my[j]]), covar,
                   min_vg_val);
  }
  if (j0 > 0) return;
  if (method != SPK_M_SK) Rs[(int64_t)n * ldr + c] = 1.0;
  if (method == SPK_M_EDK)
    for (int k = 0; k < m; ++k)
      Rs[(int64_t)(n + 1 + k) * ldr + c] = cell_drift[(int64_t)k * ldd + c];
}

// grid (row tiles x cell tiles, 1, steps); 256 threads = 4 waves, wave w
// owns cells [32 w, 32 w + 32) of the tile over its 64 rows as 4 x 2 MFMA
// 16 x 16 tiles, k in chunks of BK staged through LDS, the next chunk loaded
// into registers while the current one is multiplied.  M is column-major
// (lda), R row-major.  Blocks of one XCD take consecutive row tiles of one
// cell tile, which they then read from that XCD's L2: one block per cell
// tile that walked all row tiles read R from memory for every one of them
// and, compiled for one wave per SIMD, moved its accumulators between
// register files in every chunk (900 stations x 250 000 cells: 12.6 ms per
// step, 32 TF; now 7.8 ms, 52 TF).  Bound: FP64 MFMA issue, 77 TF measured
// with registers only.  The bounds keep 2 to 3 waves per SIMD and the
// accumulators in VGPRs.
template <int BK>
__global__ __launch_bounds__(256, BK == 8 ? 3 : 2) void k_plain_gemm(
    const double *__restrict__ M, int64_t lda, int64_t strideM,
    const double *__restrict__ R, int64_t ldr, int64_t strideR,
    const StepSc *__restrict__ sc, int p, int want_var,
    const double *__restrict__ zact, int64_t ldz, int nrt, int64_t Cs,
    double *__restrict__ part, int64_t ldq, const int *__restrict__ ccount) {
  constexpr int BM = 64, BN = 128, NT = 256;
  // 16 doubles of padding: the four 16-lane groups of a read (four k rows)
  // start 32 banks apart
  constexpr int PAD = 16;
  constexpr int AL = BM * BK / 2 / NT, BL = BN * BK / 2 / NT;
  const int sl = blockIdx.z;
  const int status = sc[sl].status, n = sc[sl].n;
  if (status) return;
  if (ccount) Cs = min(Cs, (int64_t)*ccount);
  const int lin = xcd_remap(blockIdx.x, gridDim.x);
  const int rti = lin % nrt, cti = lin / nrt;
  const int P = n + p, r0 = rti * BM;
  const int64_t c0 = cti * (int64_t)BN;
  if (r0 >= P || c0 >= Cs) return;
  M += (int64_t)sl * strideM;
  R += (int64_t)sl * strideR;
  const double *z = zact + (int64_t)sl * ldz;
  __shared__ __align__(16) double As[2][BK][BM + PAD];
  __shared__ __align__(16) double Bs[2][BK][BN + PAD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  double2 ra[AL], rb[BL];
  auto load = [&](int k0) {
#pragma unroll
    for (int q = 0; q < AL; ++q) {
      const int e = tid + q * NT;
      const int r = (e % (BM / 2)) * 2, k = e / (BM / 2);
      double2 v = {0.0, 0.0};
      // rows past P are never used but may hold stale values; a pair that
      // starts below P lies inside the column (lda is even)
      if (k0 + k < P && r0 + r < P) {
        v = *reinterpret_cast<const double2 *>(M + (r0 + r) +
                                               (int64_t)(k0 + k) * lda);
        if (r0 + r + 1 >= P) v.y = 0.0;
      }
      ra[q] = v;
    }
#pragma unroll
    for (int q = 0; q < BL; ++q) {
      const int e = tid + q * NT;
      const int c = (e % (BN / 2)) * 2, k = e / (BN / 2);
      rb[q] = k0 + k < P ? *reinterpret_cast<const double2 *>(
                               R + (int64_t)(k0 + k) * ldr + c0 + c)
                         : double2{0.0, 0.0};
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int q = 0; q < AL; ++q) {
      const int e = tid + q * NT;
      *reinterpret_cast<double2 *>(&As[buf][e / (BM / 2)]
                                      [(e % (BM / 2)) * 2]) = ra[q];
    }
#pragma unroll
    for (int q = 0; q < BL; ++q) {
      const int e = tid + q * NT;
      *reinterpret_cast<double2 *>(&Bs[buf][e / (BN / 2)]
                                      [(e % (BN / 2)) * 2]) = rb[q];
    }
  };
  p4_t acc[4][2];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = p4_t{0, 0, 0, 0};
  const int nch = (P + BK - 1) / BK;
  load(0);
  store(0);
  __syncthreads();
  for (int ch = 0; ch < nch; ++ch) {
    const int buf = ch & 1;
    if (ch + 1 < nch) load((ch + 1) * BK);
#pragma unroll
    for (int kk = 0; kk < BK / 4; ++kk) {
      const int ka = kk * 4 + lg;
      double af[4], bf[2];
#pragma unroll
      for (int t = 0; t < 4; ++t) af[t] = As[buf][ka][t * 16 + li];
#pragma unroll
      for (int t = 0; t < 2; ++t) bf[t] = Bs[buf][ka][wave * 32 + t * 16 + li];
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[a], bf[b],
                                                           acc[a][b], 0, 0, 0);
    }
    if (ch + 1 < nch) store(buf ^ 1);
    __syncthreads();
  }
  // this tile's shares: lambda.z, sum lambda, lambda.gamma + 2 mu
  double e[2] = {0.0, 0.0}, l[2] = {0.0, 0.0}, v[2] = {0.0, 0.0};
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int64_t col = c0 + wave * 32 + b * 16 + li;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = r0 + a * 16 + lg + 4 * r;
        const double w = acc[a][b][r];
        if (row < n) {
          e[b] += w * z[row];
          l[b] += w;
        }
        // row n is the multiplier mu, whose right-hand side is one
        if (want_var && row <= n && col < Cs)
          v[b] += w * (row < n ? R[(int64_t)row * ldr + col] : 2.0);
      }
    e[b] += __shfl_xor(e[b], 16, 64);
    e[b] += __shfl_xor(e[b], 32, 64);
    l[b] += __shfl_xor(l[b], 16, 64);
    l[b] += __shfl_xor(l[b], 32, 64);
    v[b] += __shfl_xor(v[b], 16, 64);
    v[b] += __shfl_xor(v[b], 32, 64);
  }
  if (lg != 0) return;
  double *q = part + ((int64_t)sl * 3 * nrt + rti) * ldq;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int64_t col = c0 + wave * 32 + b * 16 + li;
    if (col >= Cs) continue;
    q[col] = e[b];
    q[(int64_t)nrt * ldq + col] = l[b];
    if (want_var) q[(int64_t)2 * nrt * ldq + col] = v[b];
  }
}
template __global__ void k_plain_gemm<8>(
    const double *, int64_t, int64_t, const double *, int64_t, int64_t,
    const StepSc *, int, int, const double *, int64_t, int, int64_t, double *,
    int64_t, const int *);
template __global__ void k_plain_gemm<16>(
    const double *, int64_t, int64_t, const double *, int64_t, int64_t,
    const StepSc *, int, int, const double *, int64_t, int, int64_t, double *,
    int64_t, const int *);
template __global__ void k_plain_gemm<32>(
    const double *, int64_t, int64_t, const double *, int64_t, int64_t,
    const StepSc *, int, int, const double *, int64_t, int, int64_t, double *,
    int64_t, const int *);

// grid (cells / 256, steps).  The nearest station is looked for only where
// a cell of the block fails the sum-of-weights test.  cmap (optional): the
// output index of each cell.
__global__ __launch_bounds__(256) void k_plain_fin(
    const double *__restrict__ sx, const double *__restrict__ sy,
    const int32_t *__restrict__ idx, int64_t N, StepSc *__restrict__ sc,
    int p, int method, int want_var, int skm, const double *__restrict__ zact,
    int64_t ldz, const double *__restrict__ cx, const double *__restrict__ cy,
    const double *__restrict__ part, int64_t ldq, int nrt, int64_t Cs,
    double *__restrict__ est, double *__restrict__ var, int64_t ldo,
    double sum_tol, const int *__restrict__ ccount,
    const int32_t *__restrict__ cmap) {
  const int sl = blockIdx.y;
  const int status = sc[sl].status, n = sc[sl].n;
  if (status) return;
  if (ccount) Cs = min(Cs, (int64_t)*ccount);
  if (blockIdx.x * (int64_t)256 >= Cs) return;
  const int tid = threadIdx.x;
  const int64_t c = blockIdx.x * (int64_t)256 + tid;
  const bool valid = c < Cs;
  double e = 0.0, l = 1.0, v = 0.0;
  if (valid) {
    const int nt = (n + p + 63) / 64;
    const double *q = part + (int64_t)sl * 3 * nrt * ldq + c;
    l = 0.0;
    for (int t = 0; t < nt; ++t) {
      e += q[(int64_t)t * ldq];
      l += q[(int64_t)(nrt + t) * ldq];
      if (want_var) v += q[(int64_t)(2 * nrt + t) * ldq];
    }
  }
  // residual check: the weights of an OK / EDK system sum to one exactly,
  // so their sum's distance from one is rounding of the explicit inverse
  const bool ill = valid && method != SPK_M_SK && fabs(l - 1.0) > sum_tol;
  if (__ballot(ill) != 0ull && (tid & 63) == 0 &&
      !(sc[sl].flags & SPK_ST_ILLCOND))
    atomicOr(&sc[sl].flags, SPK_ST_ILLCOND);
  const double *z = zact + (int64_t)sl * ldz;
  const bool far = valid && !skm && !isclose1(l);
  int bi = 0;
  if (__syncthreads_or(far ? 1 : 0)) {
    __shared__ double2 st[256];
    __shared__ int id[256];
    const int32_t *my = idx + (int64_t)sl * N;
    const double x = valid ? cx[c] : 0.0, y = valid ? cy[c] : 0.0;
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
        const double d = dist2(x, y, st[j].x, st[j].y);
        // ties go to the lower station index (np.argmin), whatever order
        // the step's stations are compacted in
        if (d < best || (d == best && id[j] < bid)) {
          best = d;
          bi = base + j;
          bid = id[j];
        }
      }
    }
  }
  if (!valid) return;
  const int64_t oc = cmap ? (int64_t)cmap[c] : c;
  double *eo = est + (int64_t)sl * ldo;
  double *vo = var ? var + (int64_t)sl * ldo : nullptr;
  if (skm) {
    // SK with the step mean m as known mean: m + lambda^T (z - m)
    eo[oc] = e + sc[sl].mean * (1.0 - l);
  } else if (!far) {
    eo[oc] = e;
    if (want_var) vo[oc] = v;
  } else {
    eo[oc] = z[bi];
    if (want_var) vo[oc] = 0.0;
  }
}

}  // namespace spk
