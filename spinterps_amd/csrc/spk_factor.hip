// Per-step kriging systems: station compaction, covariance assembly,
// Cholesky, triangular inverse, the dual-form vectors of the batched path
// and the explicit inverse operator of the plain path.
//
// Every launch covers a whole batch of uneven systems, over (blocks, steps)
// or one workgroup per step for the small parts.  Matrices are column-major
// with a common leading dimension `ld`.
//
// Reference: interp/steps.py:170-243 (system layout), :350-371 (inverse),
// misc.py:1074-1105 (nugget-only check), interp/steps.py:276, :760-765
// (step means and interpolation flags).
#include <algorithm>

#include "spk_krige.h"

namespace spk {

// ---- step compaction -------------------------------------------------------
// Active stations (non-NaN values) of each step, in station order (or in
// the order sorder gives, a spatially compact one for the batched path), as
// interp/grps.py:57-101 forms a step's station set; the step mean over them
// (interp/steps.py:276) and the "any value >= min_var_thr" flag
// (interp/steps.py:760-765); then the step status.
__global__ __launch_bounds__(256) void k_compact(
    const double *__restrict__ vals, int64_t N, int32_t *__restrict__ idx,
    double *__restrict__ zact, int64_t ldz, StepSc *__restrict__ sc,
    const spk_vg *__restrict__ vgs, int method, double thr,
    double min_vg_val, const int32_t *__restrict__ sorder) {
  const int s = blockIdx.x;
  const double *row = vals + (int64_t)s * N;
  int32_t *my_idx = idx + (int64_t)s * N;
  double *my_z = zact + (int64_t)s * ldz;
  __shared__ int wave_cnt[4];
  __shared__ double red[256], red_abs[256];
  __shared__ int red_any[256];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int base_off = 0;
  double sum = 0.0, sabs = 0.0;
  int any = 0;
  for (int64_t b = 0; b < N; b += 256) {
    const int64_t i = (b + tid < N && sorder) ? (int64_t)sorder[b + tid]
                                               : b + tid;
    const double v = (b + tid < N) ? row[i] : NAN;
    const bool act = !isnan(v);
    const unsigned long long m = __ballot(act);
    const int pre = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) wave_cnt[wave] = __popcll(m);
    __syncthreads();
    int woff = 0;
    for (int w = 0; w < wave; ++w) woff += wave_cnt[w];
    if (act) {
      const int pos = base_off + woff + pre;
      my_idx[pos] = (int32_t)i;
      my_z[pos] = v;
      sum += v;
      sabs += fabs(v);
      any |= (v >= thr) ? 1 : 0;
    }
    const int tot = wave_cnt[0] + wave_cnt[1] + wave_cnt[2] + wave_cnt[3];
    __syncthreads();
    base_off += tot;
  }
  red[tid] = sum;
  red_abs[tid] = sabs;
  red_any[tid] = any;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) {
      red[tid] += red[tid + w];
      red_abs[tid] += red_abs[tid + w];
      red_any[tid] |= red_any[tid + w];
    }
    __syncthreads();
  }
  if (tid == 0) {
    const int n = base_off;
    StepSc &o = sc[s];
    o.n = n;
    o.mean = n > 0 ? red[0] / n : NAN;
    o.zabs = n > 0 ? red_abs[0] / n : 0.0;
    int st = 0;
    if (n == 0) {
      st = SPK_ST_NOSTNS;
    } else if (n == 1) {
      st = SPK_ST_ONESTN;
    } else if (method == SPK_M_IDW) {
      if (!red_any[0]) st = SPK_ST_MEANFILL;
    } else if (method == SPK_M_NNB) {
      st = 0;
    } else {
      const spk_vg &vg = vgs[s];
      const bool nug =
          (vg.sill_sum <= min_vg_val) || (vg.range_max_raw <= min_vg_val);
      if (!red_any[0] || nug) st = SPK_ST_MEANFILL;
    }
    o.status = st;
    o.flags = 0;
    o.planes = 0;
    o.pinv = 0;
    o.kappa = 0.0;
    o.c0 = 0.0;
    o.b = 0.0;
    o.a0 = 0.0;
    for (int k = 0; k < kMaxP; ++k) {
      o.h[k] = 0.0;
      o.dh[k] = 0.0;
    }
  }
}

// ---- system assembly ---------------------------------------------------------
// A[i, j] for i, j < n: the semivariogram sum G (OK, EDK) or the covariance
// sum (SK) of fill_vg_var_arr (pyx:146-226) at the distance of active
// stations i and j.  Coordinates are already re-centred.
__global__ __launch_bounds__(256) void k_assemble(
    const double *__restrict__ sx, const double *__restrict__ sy,
    const int32_t *__restrict__ idx, int64_t N, const StepSc *__restrict__ sc,
    const spk_vg *__restrict__ vgs, int covar_flag, double min_vg_val,
    double *__restrict__ A, int64_t ld, int64_t strideA,
    double *__restrict__ Gfull) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int tiles = (n + 63) / 64;
  const int t = blockIdx.x;
  if (t >= tiles * tiles) return;
  const int bi = t % tiles, bj = t / tiles;
  if (bi < bj) return;  // lower block triangle, mirrored on write
  __shared__ double rx[64], ry[64], cx[64], cy[64];
  __shared__ spk_vg vg;
  const int tid = threadIdx.x;
  const int32_t *my = idx + (int64_t)s * N;
  if (tid < 64) {
    const int i = bi * 64 + tid;
    rx[tid] = i < n ? sx[my[i]] : 0.0;
    ry[tid] = i < n ? sy[my[i]] : 0.0;
  } else if (tid < 128) {
    const int j = bj * 64 + tid - 64;
    cx[tid - 64] = j < n ? sx[my[j]] : 0.0;
    cy[tid - 64] = j < n ? sy[my[j]] : 0.0;
  }
  if (tid == 0) vg = vgs[s];
  __syncthreads();
  double *As = A + (int64_t)s * strideA;
  for (int e = tid; e < 64 * 64; e += 256) {
    const int r = e & 63, c = e >> 6;
    const int i = bi * 64 + r, j = bj * 64 + c;
    if (i >= n || j >= n || (bi == bj && i < j)) continue;
    const double d = dist2(rx[r], ry[r], cx[c], cy[c]);
    const double v = vg_entry(vg, d, covar_flag, min_vg_val);
    As[i + (int64_t)j * ld] = v;
    As[j + (int64_t)i * ld] = v;
    if (Gfull) {
      double *Gs = Gfull + (int64_t)s * strideA;
      Gs[i + (int64_t)j * ld] = v;
      Gs[j + (int64_t)i * ld] = v;
    }
  }
}

// ---- Cholesky ------------------------------------------------------------------
// For OK/EDK the semivariogram matrix G is first shifted to covariance form
// C = c0 - G (c0 = sum of sills for bounded models, otherwise twice the
// largest entry plus the sill sum).  The constant shift leaves the kriging
// weights unchanged because they sum to one, which is also why the
// reference's nugget (added to every entry, pyx:192-201) cancels.  Then
// C = L L^T, right-looking, in 64-wide panels: k_chol_diag factors the
// panel's diagonal block, k_chol_solve solves the rows below it,
// k_chol_trail subtracts the panel's outer product from the trailing
// triangle on FP64 MFMA.  A failed pivot marks the step SPK_ST_FAILED
// (interp/steps.py:363-384), after which its later launches return at once.
// 32-wide panels on the vector ALU read and wrote the trailing triangle
// twice as often and multiplied out of LDS at two reads per four products:
// 16 steps of up to 2 000 stations took 13 ms (shift 4.9 with one workgroup
// per step, diagonal 1.5, solve 0.6, trailing 6.2), now 2.2 (0.05, 0.7, 0.6,
// 0.8).

typedef double f4d_t __attribute__((ext_vector_type(4)));
__device__ inline f4d_t mfma64(double a, double b, f4d_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// c0 of one step, by the workgroup; every thread returns it.
__device__ inline double chol_c0(const double *As, int64_t ld, int n,
                                 const spk_vg &vg) {
  const int tid = threadIdx.x;
  __shared__ double red[256];
  bool bounded = true;
  for (int k = 0; k < vg.n; ++k) {
    const int t = vg.type[k];
    if (t == SPK_VG_RNG || t == SPK_VG_POW || t == SPK_VG_HOL)
      bounded = false;
  }
  if (bounded) return vg.sill_sum;
  double mx = 0.0;
  for (int64_t e = tid; e < (int64_t)n * n; e += 256) {
    const int i = (int)(e % n), j = (int)(e / n);
    if (i >= j) mx = fmax(mx, fabs(As[i + (int64_t)j * ld]));
  }
  red[tid] = mx;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) red[tid] = fmax(red[tid], red[tid + w]);
    __syncthreads();
  }
  return 2.0 * red[0] + fabs(vg.sill_sum);
}

// c0 of every step (grid (steps)).
__global__ __launch_bounds__(256) void k_chol_c0(const double *__restrict__ A,
                                                 int64_t ld, int64_t strideA,
                                                 StepSc *__restrict__ sc,
                                                 const spk_vg *__restrict__ vgs) {
  const int s = blockIdx.x;
  if (sc[s].status) return;
  const double c0 =
      chol_c0(A + (int64_t)s * strideA, ld, sc[s].n, vgs[s]);
  if (threadIdx.x == 0) sc[s].c0 = c0;
}

// A <- c0 - A on the lower triangle; grid (column groups, steps), block x
// takes columns x, x + gridDim.x, ...
__global__ __launch_bounds__(256) void k_chol_shift(double *__restrict__ A,
                                                    int64_t ld,
                                                    int64_t strideA,
                                                    const StepSc *__restrict__ sc) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const double c0 = sc[s].c0;
  double *As = A + (int64_t)s * strideA;
  for (int j = blockIdx.x; j < n; j += gridDim.x)
    for (int i = j + (int)threadIdx.x; i < n; i += 256)
      As[i + (int64_t)j * ld] = c0 - As[i + (int64_t)j * ld];
}

__device__ inline double lane_value(double v, int src) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)b, src);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), src);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// The panel's 64 x 64 diagonal block in LDS, 16 columns at a time: the first
// wave factors the 16 columns with row i in lane i's registers (pivots and
// multipliers by readlane, no barrier inside), then all waves update the
// columns to their right.  Bound by the chain of 64 reciprocal square roots;
// 32 columns with three barriers each took 24 us, 64 now 22 us.
// SHIFT: the whole of a system of at most 64 rows, c0 and the shift
// included.  grid (steps)
template <bool SHIFT>
__global__ __launch_bounds__(256) void k_chol_diag(
    double *__restrict__ A, int64_t ld, int64_t strideA,
    StepSc *__restrict__ sc, const spk_vg *__restrict__ vgs, int k0) {
  const int s = blockIdx.x;
  if (sc[s].status) return;
  const int n = sc[s].n;
  if (k0 >= n) return;
  const int jb = min(64, n - k0);
  double *As = A + (int64_t)s * strideA;
  const int tid = threadIdx.x, lane = tid & 63;
  __shared__ double D[64][65];  // D[column][row]
  __shared__ int fail;
  if (tid == 0) fail = 0;
  double c0 = 0.0;
  if (SHIFT) {
    c0 = chol_c0(As, ld, n, vgs[s]);
    if (tid == 0) sc[s].c0 = c0;
  }
  for (int e = tid; e < 64 * 64; e += 256) {
    const int i = e & 63, j = e >> 6;
    double v = i == j ? 1.0 : 0.0;
    if (i < jb && j < jb && i >= j) {
      v = As[(k0 + i) + (int64_t)(k0 + j) * ld];
      if (SHIFT) v = c0 - v;
    }
    D[j][i] = v;
  }
  __syncthreads();
  for (int b = 0; b < jb; b += 16) {
    if (tid < 64) {
      double a[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) a[c] = D[b + c][lane];
      bool bad = false;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const double d = lane_value(a[j], b + j);
        bad = bad || !(d > 0.0) || !isfinite(d);
        const double l = a[j] * rsqrt(d);  // d / sqrt(d) at the pivot
        a[j] = l;
#pragma unroll
        for (int c = j + 1; c < 16; ++c) a[c] -= l * lane_value(l, b + c);
      }
#pragma unroll
      for (int c = 0; c < 16; ++c) D[b + c][lane] = a[c];
      if (bad && lane == 0) fail = 1;
    }
    __syncthreads();
    if (fail) break;
    // columns b + 16 .. 63, rows from the diagonal down
    for (int c = b + 16 + (tid >> 6); c < 64; c += 4) {
      double v = D[c][lane];
#pragma unroll
      for (int j = 0; j < 16; ++j) v -= D[b + j][lane] * D[b + j][c];
      D[c][lane] = v;
    }
    __syncthreads();
  }
  if (fail) {
    if (tid == 0) sc[s].status = SPK_ST_FAILED;
    return;
  }
  for (int e = tid; e < 64 * 64; e += 256) {
    const int i = e & 63, j = e >> 6;
    if (i < jb && j < jb && i >= j)
      As[(k0 + i) + (int64_t)(k0 + j) * ld] = D[j][i];
  }
}

// Forward substitution L x = a for 64 right-hand sides, one per lane of a
// wave: 16 unknowns at a time in registers, first reduced by the earlier ones
// (kept in LDS, as many FMAs as 16-byte broadcasts of L allow), then solved
// among themselves.  Lt[q][c] = L[c][q], dinv[c] = 1 / L[c][c], a(c) the
// lane's right-hand side, done(c, x) takes the results, for the unknowns
// below `rows` (and those of its last block of 16).  The loops over the
// blocks stay rolled: fully unrolled, with all 64 unknowns in registers, the
// 35 KB of code took 50 to 78 us per launch, bound by instruction fetch; this
// takes 18 to 33.
template <typename A, typename D>
__device__ inline void wave_fwd_subst(const double (*Lt)[64],
                                      const double *dinv, double (*Xs)[64],
                                      int rows, A a, D done) {
  const int lane = threadIdx.x & 63;
#pragma unroll 1
  for (int b = 0; b < rows; b += 16) {
    double x[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) x[c] = a(b + c);
#pragma unroll 2
    for (int k = 0; k < b; ++k) {
      const double xk = Xs[k][lane];
#pragma unroll
      for (int c = 0; c < 16; ++c) x[c] -= Lt[k][b + c] * xk;
    }
#pragma unroll
    for (int c = 0; c < 16; ++c) {
#pragma unroll
      for (int q = 0; q < c; ++q) x[c] -= x[q] * Lt[b + q][b + c];
      x[c] *= dinv[b + c];
    }
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      if (b < 48) Xs[b + c][lane] = x[c];
      done(b + c, x[c]);
    }
  }
}

// rows r >= k0 + 64 solve x L_kk^T = a, one row per lane, 64 rows per
// workgroup (one wave: few rows are left in most panels);
// grid (rows below the panel / 64, steps)
__global__ __launch_bounds__(64) void k_chol_solve(double *__restrict__ A,
                                                   int64_t ld,
                                                   int64_t strideA,
                                                   const StepSc *__restrict__ sc,
                                                   int k0) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int rbase = k0 + 64 + (int)blockIdx.x * 64;
  if (rbase >= n) return;
  double *As = A + (int64_t)s * strideA;
  const int lane = threadIdx.x;
  __shared__ __align__(16) double Lt[64][64];
  __shared__ double Xs[48][64];
  __shared__ double dinv[64];
#pragma unroll 16
  for (int j = 0; j < 64; ++j)
    Lt[j][lane] = As[(k0 + lane) + (int64_t)(k0 + j) * ld];
  __syncthreads();
  dinv[lane] = 1.0 / Lt[lane][lane];
  __syncthreads();
  const int r = rbase + lane;
  const double *in = As + min(r, n - 1) + (int64_t)k0 * ld;
  double *out = As + r + (int64_t)k0 * ld;
  wave_fwd_subst(
      Lt, dinv, Xs, 64, [&](int c) { return in[(int64_t)c * ld]; },
      [&](int c, double x) {
        if (r < n) out[(int64_t)c * ld] = x;
      });
}

// Trailing triangle -= P P^T, one 64 x 64 tile per workgroup, each wave
// 32 x 32 of it as 2 x 2 MFMA tiles; the panel's fragments come straight
// from memory (16 consecutive rows per lane group).  The product is formed
// transposed, so that a lane group's results are 16 consecutive rows too.
// Bound by the triangle's read and write.  Rows from n to the tile's end lie
// inside the slab (ld is a multiple of 64); what they hold only reaches
// entries that are not stored.
// grid (tiles of the largest trailing triangle, steps): tile t = (bi, bj),
// bj <= bi, t = bi (bi + 1) / 2 + bj, of the rows / columns >= k0 + 64
__global__ __launch_bounds__(256, 2) void k_chol_trail(double *__restrict__ A,
                                                    int64_t ld,
                                                    int64_t strideA,
                                                    const StepSc *__restrict__ sc,
                                                    int k0) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int m0 = k0 + 64;
  if (m0 >= n) return;
  const int nt = (n - m0 + 63) / 64;
  const int t = blockIdx.x;
  if (t >= nt * (nt + 1) / 2) return;
  int bi = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while (bi * (bi + 1) / 2 > t) --bi;
  while ((bi + 1) * (bi + 2) / 2 <= t) ++bi;
  const int bj = t - bi * (bi + 1) / 2;
  double *As = A + (int64_t)s * strideA;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int i0 = m0 + bi * 64 + (wave & 1) * 32;
  const int j0 = m0 + bj * 64 + (wave >> 1) * 32;
  const double *Pi = As + i0 + li + (int64_t)(k0 + lg) * ld;
  const double *Pj = As + j0 + li + (int64_t)(k0 + lg) * ld;
  f4d_t acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f4d_t{0, 0, 0, 0};
#pragma unroll 8
  for (int k = 0; k < 64; k += 4) {
    const double a0 = Pj[(int64_t)k * ld], a1 = Pj[16 + (int64_t)k * ld];
    const double b0 = Pi[(int64_t)k * ld], b1 = Pi[16 + (int64_t)k * ld];
    acc[0][0] = mfma64(a0, b0, acc[0][0]);
    acc[0][1] = mfma64(a0, b1, acc[0][1]);
    acc[1][0] = mfma64(a1, b0, acc[1][0]);
    acc[1][1] = mfma64(a1, b1, acc[1][1]);
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + b * 16 + li, j = j0 + a * 16 + lg + 4 * r;
        if (i < n && i >= j) As[i + (int64_t)j * ld] -= acc[a][b][r];
      }
}

int chol_steps(hipStream_t st, double *A, int64_t ld, int64_t stride,
               StepSc *sc, const spk_vg *vgs, int shift, int64_t N, int S) {
  // systems of one panel in one launch here and below: a one-step call with
  // 3 stations and its variance takes 220 us, 241 with five launches more
  if (shift && N <= 64) {
    hipLaunchKernelGGL(k_chol_diag<true>, dim3(S), dim3(256), 0, st, A, ld,
                       stride, sc, vgs, 0);
    return check_launch("k_chol");
  }
  if (shift) {
    hipLaunchKernelGGL(k_chol_c0, dim3(S), dim3(256), 0, st,
                       (const double *)A, ld, stride, sc, vgs);
    hipLaunchKernelGGL(k_chol_shift,
                       dim3((unsigned)std::min<int64_t>(N, 256), S), dim3(256),
                       0, st, A, ld, stride, (const StepSc *)sc);
  }
  for (int k0 = 0; k0 < N; k0 += 64) {
    hipLaunchKernelGGL(k_chol_diag<false>, dim3(S), dim3(256), 0, st, A, ld,
                       stride, sc, vgs, k0);
    const int64_t nt = ceil_div(N - k0, 64) - 1;
    if (nt <= 0) break;
    hipLaunchKernelGGL(k_chol_solve, dim3((unsigned)nt, S), dim3(64), 0, st, A,
                       ld, stride, (const StepSc *)sc, k0);
    hipLaunchKernelGGL(k_chol_trail, dim3((unsigned)(nt * (nt + 1) / 2), S),
                       dim3(256), 0, st, A, ld, stride, (const StepSc *)sc,
                       k0);
  }
  return check_launch("k_chol");
}

// ---- triangular inverse ----------------------------------------------------------
// X = L^-1 (lower, zeros above the diagonal) by 64 x 64 blocks: the diagonal
// blocks are the inverses of L's, X[r, r] = inv(L_rr), and below them
// X[r, c] = X[r, r] (- sum_{c <= k < r} L[r, k] X[k, c]).  Column block c is
// a chain over r that needs only its own earlier blocks, so the column
// blocks of every step run in parallel: k_trtri_diag inverts the diagonal
// blocks (grid (blocks, steps)), then k_trtri_cols runs one column block's
// chain per workgroup (grid (blocks, steps)).  The n x n region of X is
// fully written (upper part zero).

// Lane j: column j of the block's inverse by forward substitution from the
// unit vector (the column-by-column form with two barriers per column took
// 105 us, this 21).
__global__ __launch_bounds__(64) void k_trtri_diag(
    const double *__restrict__ L, double *__restrict__ X, int64_t ld,
    int64_t stride, const StepSc *__restrict__ sc) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int r0 = blockIdx.x * 64;
  if (r0 >= n) return;
  const int rn = min(64, n - r0);
  const double *Ls = L + (int64_t)s * stride;
  double *Xs = X + (int64_t)s * stride;
  const int lane = threadIdx.x;
  __shared__ __align__(16) double Lt[64][64];
  __shared__ double Xc[48][64];
  __shared__ double T[16][65];  // results of 16 rows, [row][column]
  __shared__ double dinv[64];
  const double *Lp = Ls + r0 + min(lane, rn - 1) + (int64_t)r0 * ld;
#pragma unroll 16
  for (int j = 0; j < 64; ++j) {
    const double v = Lp[(int64_t)min(j, rn - 1) * ld];
    Lt[j][lane] = lane < rn && j < rn && lane >= j ? v : lane == j ? 1.0 : 0.0;
  }
  __syncthreads();
  dinv[lane] = 1.0 / Lt[lane][lane];
  __syncthreads();
  wave_fwd_subst(
      Lt, dinv, Xc, rn, [&](int c) { return lane == c ? 1.0 : 0.0; },
      [&](int c, double x) {
        T[c & 15][lane] = x;
        if ((c & 15) != 15) return;
        // 16 rows done: four columns per pass, 16 consecutive rows each
        __syncthreads();
        const int i = (c & ~15) + (lane & 15);
#pragma unroll 4
        for (int j = lane >> 4; j < rn; j += 4)
          if (i < rn) Xs[(r0 + i) + (int64_t)(r0 + j) * ld] = T[lane & 15][j];
        __syncthreads();
      });
}

// Products on FP64 MFMA, each wave 32 x 32 of the 64 x 64 block as 2 x 2
// tiles, formed transposed (rows: columns of X, columns: rows of X) so that
// a lane group's results are 16 consecutive rows in memory.  k in chunks of
// 32, the next chunk loaded into registers while the current one is
// multiplied out of LDS (two buffers, one barrier per chunk).  X's chunk is
// kept by columns (36 doubles apart: conflict-free writes of 32 rows and
// reads of 16 columns x 4 rows).  The longest chain (block 0) bounds a
// launch of few steps: 16 steps of up to 2 000 stations took 7.1 ms on the
// vector ALU, now 2.3 (64 hourly steps: 20.8, now 6.3).
__global__ __launch_bounds__(256, 2) void k_trtri_cols(
    const double *__restrict__ L, double *__restrict__ X, int64_t ld,
    int64_t stride, const StepSc *__restrict__ sc) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int cb = blockIdx.x;
  const int c0 = cb * 64;
  if (c0 >= n) return;
  const double *Ls = L + (int64_t)s * stride;
  double *Xs = X + (int64_t)s * stride;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
  __shared__ double La[2][32][80];  // [k][row of L]
  __shared__ double Xt[2][64][36];  // [column of X][k]
  // the sums, [column of X][row], in La's space once its chunks are read
  double (*At)[68] = reinterpret_cast<double (*)[68]>(&La[0][0][0]);
  const int nb = (n + 63) / 64;
  const int cn = min(64, n - c0);
  // the strictly-upper blocks of this column block
  for (int64_t e = tid; e < (int64_t)c0 * cn; e += 256) {
    const int i = (int)(e % c0), j = (int)(e / c0);
    Xs[i + (int64_t)(c0 + j) * ld] = 0.0;
  }
  double pa[8], pb[8];
  for (int rb = cb + 1; rb < nb; ++rb) {
    const int r0 = rb * 64;
    const int rn = min(64, n - r0);
    auto fetch = [&](int k0) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int e = tid + q * 256;
        const int r = e & 63, k = e >> 6;
        pa[q] = r < rn ? Ls[(r0 + r) + (int64_t)(k0 + k) * ld] : 0.0;
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int e = tid + q * 256;
        const int k = e & 31, c = e >> 5;
        pb[q] = c < cn ? Xs[(k0 + k) + (int64_t)(c0 + c) * ld] : 0.0;
      }
    };
    auto put = [&](int buf) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int e = tid + q * 256;
        La[buf][e >> 6][e & 63] = pa[q];
        Xt[buf][e >> 5][e & 31] = pb[q];
      }
    };
    f4d_t acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = f4d_t{0, 0, 0, 0};
    fetch(c0);
    put(0);
    __syncthreads();
    const int nch = (r0 - c0) / 32;
    for (int ch = 0; ch < nch; ++ch) {
      const int buf = ch & 1;
      if (ch + 1 < nch) fetch(c0 + (ch + 1) * 32);
#pragma unroll
      for (int kk = 0; kk < 32; kk += 4) {
        const double a0 = Xt[buf][wj + li][kk + lg];
        const double a1 = Xt[buf][wj + 16 + li][kk + lg];
        const double b0 = La[buf][kk + lg][wi + li];
        const double b1 = La[buf][kk + lg][wi + 16 + li];
        acc[0][0] = mfma64(a0, b0, acc[0][0]);
        acc[0][1] = mfma64(a0, b1, acc[0][1]);
        acc[1][0] = mfma64(a1, b0, acc[1][0]);
        acc[1][1] = mfma64(a1, b1, acc[1][1]);
      }
      if (ch + 1 < nch) put(buf ^ 1);
      __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          At[wj + a * 16 + lg + 4 * r][wi + b * 16 + li] = acc[a][b][r];
    __syncthreads();
    // X[r, c] = - X[r, r] sums; X[r, r] (zero above its diagonal) straight
    // from memory
    f4d_t out[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) out[a][b] = f4d_t{0, 0, 0, 0};
#pragma unroll 4
    for (int k = 0; k < 64; k += 4) {
      const double a0 = At[wj + li][k + lg], a1 = At[wj + 16 + li][k + lg];
      double b0 = 0.0, b1 = 0.0;
      if (k + lg < rn) {
        const double *Dp = Xs + r0 + wi + li + (int64_t)(r0 + k + lg) * ld;
        if (wi + li < rn) b0 = Dp[0];
        if (wi + 16 + li < rn) b1 = Dp[16];
      }
      out[0][0] = mfma64(a0, b0, out[0][0]);
      out[0][1] = mfma64(a0, b1, out[0][1]);
      out[1][0] = mfma64(a1, b0, out[1][0]);
      out[1][1] = mfma64(a1, b1, out[1][1]);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = wi + b * 16 + li, j = wj + a * 16 + lg + 4 * r;
          if (i < rn && j < cn)
            Xs[(r0 + i) + (int64_t)(c0 + j) * ld] = -out[a][b][r];
        }
    // the next row block reads this one's rows (same workgroup), and At
    __syncthreads();
  }
}

int trtri_steps(hipStream_t st, const double *L, double *X, int64_t ld,
                int64_t stride, const StepSc *sc, int64_t N, int S) {
  const dim3 g((unsigned)ceil_div(N, 64), S);
  hipLaunchKernelGGL(k_trtri_diag, g, dim3(64), 0, st, L, X, ld, stride, sc);
  if (N > 64)  // one diagonal block is the whole inverse
    hipLaunchKernelGGL(k_trtri_cols, g, dim3(256), 0, st, L, X, ld, stride,
                       sc);
  return check_launch("k_trtri");
}

// ---- dual-form vectors (batched path) -----------------------------------------
// With Li = L^-1:  C^-1 x = Li^T (Li x).
//   OK : w = C^-1 1, b = 1^T w, az = C^-1 z, sz = 1^T az,
//        alpha = az - w sz / b, a0 = sz / b  ->  est = k.alpha + a0
//        (the Schur complement of the Lagrange row, interp/steps.py:212-216)
//   SK : alpha = C^-1 z, w = C^-1 1 (sum of weights for the isclose test of
//        interp/steps.py:418)
//   EDK: F = [1 | S], U = Li F, W = Li^T U, B = U^T U, h = B^-1 U^T (Li z),
//        alpha = C^-1 z - W h  ->  est = k.alpha + h.[1; s_cell]
// alpha and h solve the bordered system [C F; F^T 0] [alpha; h] = [z; 0].
// Two steps of iterative refinement follow, with FP64 residuals against
// the covariances the Cholesky factorised (recomputed from the
// coordinates): r1 = z - C alpha - F h, r2 = -F^T alpha, rw = 1 - C w;
// dh = B^-1 (F^T C^-1 r1 - r2), dalpha = C^-1 r1 - W dh, dw = C^-1 rw.
// The corrections are added; the second step's are kept: k.dalpha + f.dh
// is the last change of a cell's estimate, of the size of the error left,
// which the cell kernel uses as its error indicator.
// Vectors are stored per step in V[s][0:ld] (alpha), V[s][ld:2 ld] (w),
// V[s][2 ld:3 ld] (dalpha) and V[s][3 ld:4 ld] (dw); dh in the StepSc.
__device__ inline double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Sum over the 256-thread block (all threads receive the result).
__device__ inline double block_sum(double v, double *red4) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red4[threadIdx.x >> 6] = v;
  __syncthreads();
  return red4[0] + red4[1] + red4[2] + red4[3];
}

__device__ void small_inverse(double *B, int p, double *Binv) {
  // Gauss-Jordan with partial pivoting on a p x p (p <= kMaxP) row-major.
  double a[kMaxP][2 * kMaxP];
  for (int i = 0; i < p; ++i)
    for (int j = 0; j < 2 * p; ++j)
      a[i][j] = j < p ? B[i * p + j] : (j - p == i ? 1.0 : 0.0);
  for (int c = 0; c < p; ++c) {
    int piv = c;
    for (int r = c + 1; r < p; ++r)
      if (fabs(a[r][c]) > fabs(a[piv][c])) piv = r;
    if (piv != c)
      for (int j = 0; j < 2 * p; ++j) {
        double t = a[c][j];
        a[c][j] = a[piv][j];
        a[piv][j] = t;
      }
    const double d = a[c][c];
    for (int j = 0; j < 2 * p; ++j) a[c][j] /= d;
    for (int r = 0; r < p; ++r) {
      if (r == c) continue;
      const double f = a[r][c];
      for (int j = 0; j < 2 * p; ++j) a[r][j] -= f * a[c][j];
    }
  }
  for (int i = 0; i < p; ++i)
    for (int j = 0; j < p; ++j) Binv[i * p + j] = a[i][p + j];
}

// Rows per workgroup of the triangular products L x: lane = row, the four
// waves take a quarter of the columns each, and their sums are added in
// wave order.  (One row per thread over all columns kept 16 steps of 2 000
// rows on 128 workgroups: 83 us per product, now 33; two columns 642, now
// 70.)
constexpr int kLmvRows = 64;

// This wave's share of (T X[:, r])[i], r < NR, for the block's rows i0 ..
// i0 + 63 (T lower, column-major), summed over the block's waves into red
// and returned to the first wave.
template <int NR>
__device__ inline void block_lmv(const double *__restrict__ T, int64_t ld,
                                 int n, int i0, const double *__restrict__ X,
                                 int64_t ldx, double (*red)[4][64],
                                 double *acc) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = i0 + lane;
  const double *Ti = T + min(i, n - 1);
  const int kend = min(n, i0 + kLmvRows);
  const int len = (kend + 3) / 4;
  const int k1 = min(kend, (wave + 1) * len);
#pragma unroll
  for (int r = 0; r < NR; ++r) acc[r] = 0.0;
#pragma unroll 8
  for (int k = wave * len; k < k1; ++k) {
    // (what lies above the diagonal is loaded and not used)
    const double t = Ti[(int64_t)k * ld];
    const double l = k <= i ? t : 0.0;
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] += l * X[k + (int64_t)r * ldx];
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) red[r][wave][lane] = acc[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < NR; ++r)
    acc[r] = red[r][0][lane] + red[r][1][lane] + red[r][2][lane] +
             red[r][3][lane];
}

// ---- condition estimate over (block, step) workgroups --------------------------
// kappa = lambda_max(C) lambda_max(C^-1) by power iteration on C = Lc Lc^T
// (which 0, Lc the Cholesky factor) and C^-1 = Li^T Li (which 1), 12 rounds
// each, Rayleigh quotients; the iterate x and u = T^T x or T x are the first
// two scratch columns of the step's T0 (X and U of k_dual).  Launch order
// per which: k_kap_start, then 12 x (k_kap_norm, product into u,
// k_kap_rq, product back into x); then k_kap_flags.  The products run over
// (row blocks, steps), 64 rows per workgroup (k_kap_lmv, y = T x) or one
// column per wave (k_kap_umv, y = T^T x), and the norms as one workgroup per
// step.
__device__ inline double *kap_x(double *T0, int64_t ldt, int s) {
  return T0 + (int64_t)s * ldt * kT0Cols;
}
__device__ inline double *kap_u(double *T0, int64_t ldt, int s) {
  return kap_x(T0, ldt, s) + ldt * (kMaxP + 1);
}

// grid (steps)
__global__ __launch_bounds__(256) void k_kap_start(const StepSc *__restrict__ sc,
                                                   double *__restrict__ T0,
                                                   int64_t ldt, int which) {
  const int s = blockIdx.x;
  if (sc[s].status) return;
  const int n = sc[s].n;
  double *X = kap_x(T0, ldt, s);
  for (int i = threadIdx.x; i < n; i += 256) {
    // fixed start vector with both smooth and oscillating parts
    const unsigned h = (unsigned)i * 2654435761u;
    X[i] = 1.0 + 0.5 * (double)((h >> 8) & 0xffff) / 65536.0 -
           (which ? 0.5 * (double)(i & 1) : 0.0);
  }
}

// x /= |x|; grid (steps)
__global__ __launch_bounds__(256) void k_kap_norm(const StepSc *__restrict__ sc,
                                                  double *__restrict__ T0,
                                                  int64_t ldt) {
  const int s = blockIdx.x;
  if (sc[s].status) return;
  const int n = sc[s].n;
  double *X = kap_x(T0, ldt, s);
  __shared__ double red4[4];
  const int tid = threadIdx.x;
  double nv = 0.0;
  for (int i = tid; i < n; i += 256) nv += X[i] * X[i];
  nv = block_sum(nv, red4);
  const double inv = 1.0 / sqrt(nv);
  for (int i = tid; i < n; i += 256) X[i] *= inv;
}

// lam[2 s + which] = |u|^2; grid (steps)
__global__ __launch_bounds__(256) void k_kap_rq(const StepSc *__restrict__ sc,
                                                double *__restrict__ T0,
                                                int64_t ldt,
                                                double *__restrict__ lam,
                                                int which) {
  const int s = blockIdx.x;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const double *U = kap_u(T0, ldt, s);
  __shared__ double red4[4];
  double q = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) q += U[i] * U[i];
  q = block_sum(q, red4);
  if (threadIdx.x == 0) lam[2 * s + which] = q;
}

// y = T v (T lower, column-major, ld), v and y the step's x / u columns
// (to_u: v = x, y = u; else v = u, y = x); grid (ceil(n_max / 64), steps)
__global__ __launch_bounds__(256) void k_kap_lmv(const double *__restrict__ T,
                                                 int64_t ld, int64_t stride,
                                                 const StepSc *__restrict__ sc,
                                                 double *__restrict__ T0,
                                                 int64_t ldt, int to_u) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int i0 = blockIdx.x * kLmvRows;
  if (i0 >= n) return;
  const double *v = to_u ? kap_x(T0, ldt, s) : kap_u(T0, ldt, s);
  double *y = to_u ? kap_u(T0, ldt, s) : kap_x(T0, ldt, s);
  __shared__ double red[1][4][64];
  double acc[1];
  block_lmv<1>(T + (int64_t)s * stride, ld, n, i0, v, 0, red, acc);
  if (threadIdx.x < 64 && i0 + (int)threadIdx.x < n) y[i0 + threadIdx.x] = acc[0];
}

// y = T^T v, one wave per entry k (lanes over rows i >= k);
// grid (ceil(n_max / 4), steps)
__global__ __launch_bounds__(256) void k_kap_umv(const double *__restrict__ T,
                                                 int64_t ld, int64_t stride,
                                                 const StepSc *__restrict__ sc,
                                                 double *__restrict__ T0,
                                                 int64_t ldt, int to_u) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int lane = threadIdx.x & 63;
  const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (k >= n) return;
  const double *Ts = T + (int64_t)s * stride;
  const double *v = to_u ? kap_x(T0, ldt, s) : kap_u(T0, ldt, s);
  double *y = to_u ? kap_u(T0, ldt, s) : kap_x(T0, ldt, s);
  double acc = 0.0;
#pragma unroll 4
  for (int i = k + lane; i < n; i += 64) {
    const double l = Ts[i + (int64_t)k * ld];
    acc += l * v[i];
  }
  const double r = wave_sum(acc);
  if (lane == 0) y[k] = r;
}

// kappa and the step's precision flags; grid (steps), one thread
__global__ void k_kap_flags(StepSc *__restrict__ sc,
                            const double *__restrict__ lam,
                            const spk_vg *__restrict__ vgs,
                            double fp64var_thr, double fp64var_thr_gau,
                            double int8var_thr) {
  const int s = blockIdx.x;
  if (threadIdx.x != 0 || sc[s].status) return;
  const double kap = lam[2 * s] * lam[2 * s + 1];
  sc[s].kappa = kap;
  int fl = 0;
  if (!(kap <= 1e12)) fl |= SPK_ST_ILLCOND;
  bool gau = false;
  for (int k = 0; k < vgs[s].n; ++k) gau |= vgs[s].type[k] == SPK_VG_GAU;
  // above the FP32 limit: exact int8 plane products up to the int8
  // limit, FP64 beyond it
  int planes = 0;
  if (!(kap <= (gau ? fp64var_thr_gau : fp64var_thr))) {
    if (kap <= int8var_thr)
      planes = kap <= kInt8Deep ? 5 : 6;
    else
      fl |= SPK_ST_FP64VAR;
  }
  if (planes) fl |= SPK_ST_INT8VAR;
  sc[s].flags = fl;
  sc[s].planes = planes;
}

// ---- dual vectors and refinement over (block, step) workgroups ----------------
// Per step, with T0 holding X, U (kMaxP + 1 columns each), R2, Y2, Z2 (two
// each) and the per-step scratch ds (kDualSc doubles: G, Bi, hcoef, hcur,
// dhs):
//   k_dual_rhs   X = [F z]                                    (steps)
//   k_dual_lmv   U = Li X            (p + 1 columns)          (row blocks, steps)
//   k_dual_umv   X = Li^T U = C^-1 [F z]                      (column groups, steps)
//   k_dual_mid   G = U^T U, Bi = (U_F^T U_F)^-1, h, alpha, w  (steps)
//   then twice: k_dual_resid (r1 = z - C alpha - F h, rw = 1 - C w;
//   row blocks, steps), k_dual_lmv / k_dual_umv on [r1 rw], k_dual_upd
//   (the corrections of h, alpha and w; steps); then k_dual_fin (steps).
constexpr int kDsG = 0;                                  // (p+1)^2
constexpr int kDsBi = kDsG + (kMaxP + 1) * (kMaxP + 1);  // p^2
constexpr int kDsH = kDsBi + kMaxP * kMaxP;              // hcoef
constexpr int kDsHc = kDsH + kMaxP;                      // hcur
constexpr int kDsDh = kDsHc + kMaxP;                     // dhs

struct DualPtrs {
  double *X, *U, *R2, *Y2, *Z2, *alpha, *w, *dalpha, *dw, *ds;
};
__device__ inline DualPtrs dual_ptrs(double *T0, int64_t ldt, double *V,
                                     int64_t ldv, double *DS, int s) {
  DualPtrs d;
  d.X = T0 + (int64_t)s * ldt * kT0Cols;
  d.U = d.X + ldt * (kMaxP + 1);
  d.R2 = d.U + ldt * (kMaxP + 1);  // residuals r1, rw
  d.Y2 = d.R2 + 2 * ldt;           // Li [r1 rw]
  d.Z2 = d.Y2 + 2 * ldt;           // C^-1 [r1 rw]
  d.alpha = V + (int64_t)s * ldv;
  d.w = d.alpha + ldt;
  d.dalpha = d.w + ldt;
  d.dw = d.dalpha + ldt;
  d.ds = DS + (int64_t)s * kDualSc;
  return d;
}

// X columns: 0..p-1 = F (ones, drifts), p = z; grid (steps)
__global__ __launch_bounds__(256) void k_dual_rhs(
    const StepSc *__restrict__ sc, const double *__restrict__ zact,
    int64_t ldz, const int32_t *__restrict__ idx, int64_t N,
    const double *__restrict__ stn_drift, int m, int method,
    double *__restrict__ T0, int64_t ldt) {
  const int s = blockIdx.x;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const double *z = zact + (int64_t)s * ldz;
  const int32_t *my = idx + (int64_t)s * N;
  double *X = T0 + (int64_t)s * ldt * kT0Cols;
  const int p = (method == SPK_M_EDK) ? 1 + m : 1;
  for (int i = threadIdx.x; i < n; i += 256) {
    X[i] = 1.0;
    if (method == SPK_M_EDK)
      for (int k = 0; k < m; ++k)
        X[i + (int64_t)(1 + k) * ldt] = stn_drift[(int64_t)my[i] * m + k];
    X[i + (int64_t)p * ldt] = z[i];
  }
}

// column offsets in T0 of the products' operands (col: 0 X, 1 U, 2 R2,
// 3 Y2, 4 Z2)
__device__ inline double *t0_col(double *T0, int64_t ldt, int s, int col) {
  double *X = T0 + (int64_t)s * ldt * kT0Cols;
  switch (col) {
    case 0: return X;
    case 1: return X + ldt * (kMaxP + 1);
    case 2: return X + 2 * ldt * (kMaxP + 1);
    case 3: return X + 2 * ldt * (kMaxP + 1) + 2 * ldt;
    default: return X + 2 * ldt * (kMaxP + 1) + 4 * ldt;
  }
}

// Y[:, r] = Li X[:, r] (r < nr), 64 rows per workgroup; grid (ceil(n_max /
// 64), steps)
__global__ __launch_bounds__(256) void k_dual_lmv(
    const double *__restrict__ Li, int64_t ld, int64_t stride,
    const StepSc *__restrict__ sc, double *__restrict__ T0, int64_t ldt,
    int src, int dst, int nr) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int i0 = blockIdx.x * kLmvRows;
  if (i0 >= n) return;
  const double *L = Li + (int64_t)s * stride;
  const double *X = t0_col(T0, ldt, s, src);
  double *Y = t0_col(T0, ldt, s, dst);
  __shared__ double red[2][4][64];
  const int i = i0 + (int)threadIdx.x;
  // two columns at a time ([1 z] and [r1 rw] are two)
  for (int r = 0; r < nr; r += 2) {
    double acc[2];
    if (r > 0) __syncthreads();
    if (r + 1 < nr)
      block_lmv<2>(L, ld, n, i0, X + (int64_t)r * ldt, ldt, red, acc);
    else
      block_lmv<1>(L, ld, n, i0, X + (int64_t)r * ldt, ldt, red, acc);
    if (threadIdx.x < 64 && i < n) {
      Y[i + (int64_t)r * ldt] = acc[0];
      if (r + 1 < nr) Y[i + (int64_t)(r + 1) * ldt] = acc[1];
    }
  }
}

// Y[:, r] = Li^T X[:, r], one wave per output entry (lanes over rows);
// grid (ceil(n_max / 4), steps)
__global__ __launch_bounds__(256) void k_dual_umv(
    const double *__restrict__ Li, int64_t ld, int64_t stride,
    const StepSc *__restrict__ sc, double *__restrict__ T0, int64_t ldt,
    int src, int dst, int nr) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int lane = threadIdx.x & 63;
  const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (k >= n) return;
  const double *L = Li + (int64_t)s * stride;
  const double *X = t0_col(T0, ldt, s, src);
  double *Y = t0_col(T0, ldt, s, dst);
  double acc[kMaxP + 1];
  for (int r = 0; r < nr; ++r) acc[r] = 0.0;
#pragma unroll 4
  for (int i = k + lane; i < n; i += 64) {
    const double l = L[i + (int64_t)k * ld];
    for (int r = 0; r < nr; ++r) acc[r] += l * X[i + (int64_t)r * ldt];
  }
  for (int r = 0; r < nr; ++r) {
    const double v = wave_sum(acc[r]);
    if (lane == 0) Y[k + (int64_t)r * ldt] = v;
  }
}

// G = U^T U (a, b <= p: B = U_F^T U_F, g = U_F^T U_z), Bi = B^-1, the
// Schur coefficients h = Bi g, alpha = C^-1 z - C^-1 F h, w = C^-1 1;
// grid (steps)
__global__ __launch_bounds__(256) void k_dual_mid(
    const StepSc *__restrict__ sc, int m, int method, double *__restrict__ T0,
    int64_t ldt, double *__restrict__ V, int64_t ldv, double *__restrict__ DS) {
  const int s = blockIdx.x;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const DualPtrs d = dual_ptrs(T0, ldt, V, ldv, DS, s);
  const int p = (method == SPK_M_EDK) ? 1 + m : 1;
  const int tid = threadIdx.x;
  __shared__ double G[(kMaxP + 1) * (kMaxP + 1)];
  for (int e = tid >> 6; e < (p + 1) * (p + 1); e += 4) {
    const int a = e / (p + 1), b = e % (p + 1);
    double acc = 0.0;
    for (int i = (tid & 63); i < n; i += 64)
      acc += d.U[i + (int64_t)a * ldt] * d.U[i + (int64_t)b * ldt];
    acc = wave_sum(acc);
    if ((tid & 63) == 0) G[e] = acc;
  }
  __syncthreads();
  __shared__ double hcoef[kMaxP];
  __shared__ double Bi[kMaxP * kMaxP];
  if (tid == 0) {
    double B[kMaxP * kMaxP];
    for (int a = 0; a < p; ++a)
      for (int b = 0; b < p; ++b) B[a * p + b] = G[a * (p + 1) + b];
    if (method == SPK_M_SK) {
      // no constraint rows: alpha = C^-1 z, w = C^-1 1
      hcoef[0] = 0.0;
    } else {
      small_inverse(B, p, Bi);
      for (int a = 0; a < p; ++a) {
        double v = 0.0;
        for (int b = 0; b < p; ++b) v += Bi[a * p + b] * G[b * (p + 1) + p];
        hcoef[a] = v;
      }
    }
    for (int e = 0; e < (p + 1) * (p + 1); ++e) d.ds[kDsG + e] = G[e];
    if (method != SPK_M_SK)
      for (int e = 0; e < p * p; ++e) d.ds[kDsBi + e] = Bi[e];
    for (int a = 0; a < kMaxP; ++a) {
      d.ds[kDsH + a] = a < p ? hcoef[a] : 0.0;
      d.ds[kDsHc + a] = a < p ? hcoef[a] : 0.0;
    }
  }
  __syncthreads();
  for (int i = tid; i < n; i += 256) {
    double a = d.X[i + (int64_t)p * ldt];
    if (method != SPK_M_SK)
      for (int k = 0; k < p; ++k) a -= d.X[i + (int64_t)k * ldt] * hcoef[k];
    d.alpha[i] = a;
    d.w[i] = d.X[i];
  }
}

// ---- iterative refinement with FP64 residuals ------------------------------
// r1 = z - C alpha - F h, rw = 1 - C w, with C the covariances the
// Cholesky factorised: c0 - gamma (OK, EDK) or the covariance sum (SK),
// recomputed from the re-centred coordinates with the same arithmetic.
// Two steps: the first removes the error of the explicit-inverse solve,
// the second's correction is of the size of the error left, which the
// cell kernel turns into each cell's error indicator.
// 64 rows per workgroup, a lane per row, each wave a quarter of the stations
// of every pass of 256; the waves' sums are added in wave order (one row per
// thread over all stations took 1.3 ms for 16 steps of up to 2 000 rows,
// this 0.37).
// grid (ceil(n_max / 64), steps).
__global__ __launch_bounds__(256) void k_dual_resid(
    const StepSc *__restrict__ sc, const double *__restrict__ zact,
    int64_t ldz, const int32_t *__restrict__ idx, int64_t N,
    const double *__restrict__ stn_drift, int m, int method,
    double *__restrict__ T0, int64_t ldt, double *__restrict__ V, int64_t ldv,
    double *__restrict__ DS, const spk_vg *__restrict__ vgs, double min_vg_val,
    const double *__restrict__ sx, const double *__restrict__ sy) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int i0 = blockIdx.x * kLmvRows;
  if (i0 >= n) return;
  const DualPtrs d = dual_ptrs(T0, ldt, V, ldv, DS, s);
  const double *z = zact + (int64_t)s * ldz;
  const int32_t *my = idx + (int64_t)s * N;
  const int p = (method == SPK_M_EDK) ? 1 + m : 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  __shared__ double stx[256], sty[256], sal[256], sw[256];
  __shared__ double red[2][4][64];
  __shared__ spk_vg vg;
  if (tid == 0) vg = vgs[s];
  const bool sk = method == SPK_M_SK;
  const double c0 = sc[s].c0;
  const int i = i0 + lane;
  double xi = 0.0, yi = 0.0;
  if (i < n) {
    xi = sx[my[i]];
    yi = sy[my[i]];
  }
  double ca = 0.0, cw = 0.0;
  for (int j0 = 0; j0 < n; j0 += 256) {
    __syncthreads();
    if (j0 + tid < n) {
      const int g = my[j0 + tid];
      stx[tid] = sx[g];
      sty[tid] = sy[g];
      sal[tid] = d.alpha[j0 + tid];
      sw[tid] = d.w[j0 + tid];
    }
    __syncthreads();
    const int j1 = min(wave * 64 + 64, n - j0);
    for (int j = wave * 64; j < j1; ++j) {
      const double dd = dist2(xi, yi, stx[j], sty[j]);
      const double e = vg_entry(vg, dd, sk ? 1 : 0, min_vg_val);
      const double c = sk ? e : c0 - e;
      ca += c * sal[j];
      cw += c * sw[j];
    }
  }
  red[0][wave][lane] = ca;
  red[1][wave][lane] = cw;
  __syncthreads();
  if (wave == 0 && i < n) {
    ca = red[0][0][lane] + red[0][1][lane] + red[0][2][lane] + red[0][3][lane];
    cw = red[1][0][lane] + red[1][1][lane] + red[1][2][lane] + red[1][3][lane];
    double r1 = z[i] - ca;
    if (!sk) {
      r1 -= d.ds[kDsHc + 0];
      for (int k = 1; k < p; ++k)
        r1 -= stn_drift[(int64_t)my[i] * m + (k - 1)] * d.ds[kDsHc + k];
    }
    d.R2[i] = r1;
    d.R2[i + ldt] = 1.0 - cw;
  }
}

// gF[a] = U_F[:, a] . (Li r1) = F^T C^-1 r1, r2[a] = -F[:, a] . alpha, the
// corrections dh = Bi (gF - r2), alpha += Z2[:, 0] - C^-1 F dh,
// w += Z2[:, 1]; grid (steps)
__global__ __launch_bounds__(256) void k_dual_upd(
    const StepSc *__restrict__ sc, const int32_t *__restrict__ idx, int64_t N,
    const double *__restrict__ stn_drift, int m, int method,
    double *__restrict__ T0, int64_t ldt, double *__restrict__ V, int64_t ldv,
    double *__restrict__ DS) {
  const int s = blockIdx.x;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const DualPtrs d = dual_ptrs(T0, ldt, V, ldv, DS, s);
  const int32_t *my = idx + (int64_t)s * N;
  const int p = (method == SPK_M_EDK) ? 1 + m : 1;
  const int tid = threadIdx.x;
  const bool sk = method == SPK_M_SK;
  __shared__ double gF[kMaxP], r2s[kMaxP], dhs[kMaxP];
  if (!sk) {
    for (int a = tid >> 6; a < 2 * p; a += 4) {
      double acc = 0.0;
      const int col = a < p ? a : a - p;
      for (int i = (tid & 63); i < n; i += 64) {
        if (a < p) {
          acc += d.U[i + (int64_t)col * ldt] * d.Y2[i];
        } else {
          const double f =
              col == 0 ? 1.0 : stn_drift[(int64_t)my[i] * m + (col - 1)];
          acc -= f * d.alpha[i];
        }
      }
      acc = wave_sum(acc);
      if ((tid & 63) == 0) {
        if (a < p)
          gF[col] = acc;
        else
          r2s[col] = acc;
      }
    }
  }
  __syncthreads();
  if (tid == 0) {
    for (int a = 0; a < kMaxP; ++a) dhs[a] = 0.0;
    if (!sk)
      for (int a = 0; a < p; ++a) {
        double v = 0.0;
        for (int b = 0; b < p; ++b)
          v += d.ds[kDsBi + a * p + b] * (gF[b] - r2s[b]);
        dhs[a] = v;
      }
  }
  __syncthreads();
  for (int i = tid; i < n; i += 256) {
    double da = d.Z2[i];
    if (!sk)
      for (int k = 0; k < p; ++k) da -= d.X[i + (int64_t)k * ldt] * dhs[k];
    const double dwi = d.Z2[i + ldt];
    d.alpha[i] += da;
    d.w[i] += dwi;
    d.dalpha[i] = da;
    d.dw[i] = dwi;
  }
  if (tid < p) d.ds[kDsHc + tid] += dhs[tid];
  if (tid < kMaxP) d.ds[kDsDh + tid] = dhs[tid];
}

// the step record's dual-form terms; grid (steps)
__global__ void k_dual_fin(StepSc *__restrict__ sc, int m, int method,
                           const double *__restrict__ DS) {
  const int s = blockIdx.x;
  if (threadIdx.x != 0 || sc[s].status) return;
  const double *ds = DS + (int64_t)s * kDualSc;
  const int p = (method == SPK_M_EDK) ? 1 + m : 1;
  const bool sk = method == SPK_M_SK;
  StepSc &o = sc[s];
  o.b = ds[kDsG + 0];  // 1^T C^-1 1
  for (int a = 0; a < p; ++a) {
    o.h[a] = ds[kDsHc + a];
    o.dh[a] = ds[kDsDh + a];
  }
  o.a0 = sk ? 0.0 : ds[kDsHc + 0];
}

// ---- explicit K^-1 for the plain path -------------------------------------------
// Cinv = Li^T Li; W = Cinv F; B = F^T W; Q = W B^-1; P = Cinv - Q W^T.
// The reference's K = [[G, F], [F^T, 0]] with G = c0 11^T - C has the
// inverse [[-P, Q], [Q^T, B^-1 - c0 e0 e0^T]], written to M (ld rows).
// SK has no constraint rows: M = Cinv.
// Launches over (tiles or row blocks, steps): k_minv_tiles, k_minv_w,
// k_minv_mid, k_minv_fin (minv_steps; systems of one tile: k_minv_small).  One workgroup per step for all of it
// took 11.8 ms for systems of 900 rows; the four take 0.24 ms for seven.

// Cinv[i, j] = sum over k >= i of Li[k, i] Li[k, j], a 64 x 64 tile (bi >=
// bj) per workgroup and its mirror image, on FP64 MFMA (32 x 32 per wave).
// Both operands are read down columns of Li and kept by columns in LDS (36
// doubles apart).  grid (tiles of the lower triangle, steps)
__device__ inline void minv_tile(const double *L, int64_t ld, int n, int bi,
                                 int bj, double *Ms) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int wi = (wave & 1) * 32, wj = (wave >> 1) * 32;
  __shared__ double Ti[2][64][36], Tj[2][64][36];  // [column][k]
  double pi_[8], pj_[8];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = tid + q * 256;
      const int k = k0 + (e & 31), c = e >> 5;
      pi_[q] = k < n && bi * 64 + c < n
                   ? L[k + (int64_t)(bi * 64 + c) * ld] : 0.0;
      pj_[q] = k < n && bj * 64 + c < n
                   ? L[k + (int64_t)(bj * 64 + c) * ld] : 0.0;
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int e = tid + q * 256;
      Ti[buf][e >> 5][e & 31] = pi_[q];
      Tj[buf][e >> 5][e & 31] = pj_[q];
    }
  };
  f4d_t acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = f4d_t{0, 0, 0, 0};
  fetch(bi * 64);
  put(0);
  __syncthreads();
  const int nch = (n - bi * 64 + 31) / 32;
  for (int ch = 0; ch < nch; ++ch) {
    const int buf = ch & 1;
    if (ch + 1 < nch) fetch(bi * 64 + (ch + 1) * 32);
#pragma unroll
    for (int kk = 0; kk < 32; kk += 4) {
      const double a0 = Tj[buf][wj + li][kk + lg];
      const double a1 = Tj[buf][wj + 16 + li][kk + lg];
      const double b0 = Ti[buf][wi + li][kk + lg];
      const double b1 = Ti[buf][wi + 16 + li][kk + lg];
      acc[0][0] = mfma64(a0, b0, acc[0][0]);
      acc[0][1] = mfma64(a0, b1, acc[0][1]);
      acc[1][0] = mfma64(a1, b0, acc[1][0]);
      acc[1][1] = mfma64(a1, b1, acc[1][1]);
    }
    if (ch + 1 < nch) put(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = bi * 64 + wi + b * 16 + li;
        const int j = bj * 64 + wj + a * 16 + lg + 4 * r;
        if (i < n && j < n) {
          Ms[i + (int64_t)j * ld] = acc[a][b][r];
          Ms[j + (int64_t)i * ld] = acc[a][b][r];
        }
      }
}
__global__ __launch_bounds__(256, 2) void k_minv_tiles(
    const double *__restrict__ Li, int64_t ld, int64_t stride,
    const StepSc *__restrict__ sc, double *__restrict__ M) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int nb = (n + 63) / 64;
  const int t = blockIdx.x;
  if (t >= nb * (nb + 1) / 2) return;
  int bi = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
  while (bi * (bi + 1) / 2 > t) --bi;
  while ((bi + 1) * (bi + 2) / 2 <= t) ++bi;
  minv_tile(Li + (int64_t)s * stride, ld, n, bi, t - bi * (bi + 1) / 2,
            M + (int64_t)s * stride);
}

// W = Cinv F (columns 0 .. p-1 of the step's work area T0), 64 rows per
// workgroup, each wave a quarter of the columns; grid (ceil(n_max / 64),
// steps)
__device__ inline void minv_w(const double *Ms, int64_t ld, int n, int i0,
                              const int32_t *my, const double *stn_drift,
                              int m, int p, double *W, int64_t ldt) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = min(i0 + lane, n - 1);
  __shared__ double red[kMaxP][4][64];
  double acc[kMaxP];
#pragma unroll
  for (int r = 0; r < kMaxP; ++r) acc[r] = 0.0;
  const int len = (n + 3) / 4;
  const int k1 = min(n, (wave + 1) * len);
  for (int k = wave * len; k < k1; ++k) {
    const double c = Ms[i + (int64_t)k * ld];
    acc[0] += c;
#pragma unroll
    for (int r = 1; r < kMaxP; ++r)
      if (r < p) acc[r] += c * stn_drift[(int64_t)my[k] * m + (r - 1)];
  }
#pragma unroll
  for (int r = 0; r < kMaxP; ++r) red[r][wave][lane] = acc[r];
  __syncthreads();
  for (int r = wave; r < p; r += 4)
    if (i0 + lane < n)
      W[i0 + lane + (int64_t)r * ldt] = red[r][0][lane] + red[r][1][lane] +
                                        red[r][2][lane] + red[r][3][lane];
}
__global__ __launch_bounds__(256) void k_minv_w(
    const double *__restrict__ M, int64_t ld, int64_t stride,
    const StepSc *__restrict__ sc, const int32_t *__restrict__ idx, int64_t N,
    const double *__restrict__ stn_drift, int m, int p,
    double *__restrict__ T0, int64_t ldt) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const int i0 = blockIdx.x * 64;
  if (i0 >= n) return;
  minv_w(M + (int64_t)s * stride, ld, n, i0, idx + (int64_t)s * N, stn_drift,
         m, p, T0 + (int64_t)s * ldt * kT0Cols, ldt);
}

// The condition estimate max diag(Cinv) max diag(C), then B = F^T W, its
// inverse (M's corner) and Q = W B^-1 (columns p .. 2p-1 of T0); grid
// (steps)
__device__ inline void minv_mid(double *Ms, int64_t ld, StepSc *st,
                                const int32_t *my, const double *stn_drift,
                                int m, int method, int p, double *W,
                                int64_t ldt, const spk_vg &vg,
                                double min_vg_val) {
  const int n = st->n;
  const int tid = threadIdx.x;
  __shared__ double red[256];
  double mx = 0.0;
  for (int i = tid; i < n; i += 256) mx = fmax(mx, Ms[i + (int64_t)i * ld]);
  red[tid] = mx;
  __syncthreads();
  for (int w2 = 128; w2 > 0; w2 >>= 1) {
    if (tid < w2) red[tid] = fmax(red[tid], red[tid + w2]);
    __syncthreads();
  }
  if (tid == 0) {
    const double cii = (method == SPK_M_SK)
                           ? vg_entry(vg, 0.0, 1, min_vg_val)
                           : st->c0 - vg_entry(vg, 0.0, 0, min_vg_val);
    const double kap = red[0] * fabs(cii);
    st->kappa = kap;
    st->flags = (kap <= 1e12) ? 0 : SPK_ST_ILLCOND;
  }
  if (method == SPK_M_SK) return;
  __shared__ double Bs[kMaxP * kMaxP], Bi[kMaxP * kMaxP];
  for (int e = tid >> 6; e < p * p; e += 4) {
    const int a = e / p, b = e % p;
    double acc = 0.0;
    for (int i = (tid & 63); i < n; i += 64) {
      const double fa = a == 0 ? 1.0 : stn_drift[(int64_t)my[i] * m + a - 1];
      acc += fa * W[i + (int64_t)b * ldt];
    }
    acc = wave_sum(acc);
    if ((tid & 63) == 0) Bs[e] = acc;
  }
  __syncthreads();
  if (tid == 0) small_inverse(Bs, p, Bi);
  __syncthreads();
  double *Q = W + (int64_t)p * ldt;
  for (int i = tid; i < n; i += 256)
    for (int a = 0; a < p; ++a) {
      double v = 0.0;
      for (int b = 0; b < p; ++b) v += W[i + (int64_t)b * ldt] * Bi[b * p + a];
      Q[i + (int64_t)a * ldt] = v;
    }
  if (tid < p * p) {
    const int a = tid / p, b = tid % p;
    Ms[(n + a) + (int64_t)(n + b) * ld] =
        Bi[a * p + b] - ((a == 0 && b == 0) ? st->c0 : 0.0);
  }
}
__global__ __launch_bounds__(256) void k_minv_mid(
    double *__restrict__ M, int64_t ld, int64_t stride,
    StepSc *__restrict__ sc, const int32_t *__restrict__ idx, int64_t N,
    const double *__restrict__ stn_drift, int m, int method, int p,
    double *__restrict__ T0, int64_t ldt, const spk_vg *__restrict__ vgs,
    double min_vg_val) {
  const int s = blockIdx.x;
  if (sc[s].status) return;
  minv_mid(M + (int64_t)s * stride, ld, sc + s, idx + (int64_t)s * N,
           stn_drift, m, method, p, T0 + (int64_t)s * ldt * kT0Cols, ldt,
           vgs[s], min_vg_val);
}

// M <- -(Cinv - Q W^T) and the border rows; grid (column groups, steps),
// block x takes columns x, x + gridDim.x, ...
__device__ inline void minv_fin(double *Ms, int64_t ld, int n, int p,
                                const double *W, int64_t ldt) {
  const double *Q = W + (int64_t)p * ldt;
  for (int j = blockIdx.x; j < n; j += gridDim.x) {
    for (int i = threadIdx.x; i < n; i += 256) {
      double v = Ms[i + (int64_t)j * ld];
      for (int a = 0; a < p; ++a)
        v -= Q[i + (int64_t)a * ldt] * W[j + (int64_t)a * ldt];
      Ms[i + (int64_t)j * ld] = -v;
    }
    if ((int)threadIdx.x < p) {
      const int a = threadIdx.x;
      const double q = Q[j + (int64_t)a * ldt];
      Ms[j + (int64_t)(n + a) * ld] = q;
      Ms[(n + a) + (int64_t)j * ld] = q;
    }
  }
}
__global__ __launch_bounds__(256) void k_minv_fin(
    double *__restrict__ M, int64_t ld, int64_t stride,
    const StepSc *__restrict__ sc, int p, const double *__restrict__ T0,
    int64_t ldt) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  minv_fin(M + (int64_t)s * stride, ld, sc[s].n, p,
           T0 + (int64_t)s * ldt * kT0Cols, ldt);
}

// All of it for systems of one tile (n <= 64); grid (1, steps)
__global__ __launch_bounds__(256, 2) void k_minv_small(
    const double *Li, int64_t ld, int64_t stride, StepSc *sc,
    const int32_t *idx, int64_t N, const double *stn_drift, int m, int method,
    int p, double *M, double *T0, int64_t ldt, const spk_vg *vgs,
    double min_vg_val) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  double *Ms = M + (int64_t)s * stride;
  double *W = T0 + (int64_t)s * ldt * kT0Cols;
  const int32_t *my = idx + (int64_t)s * N;
  minv_tile(Li + (int64_t)s * stride, ld, n, 0, 0, Ms);
  __syncthreads();
  if (p > 0) minv_w(Ms, ld, n, 0, my, stn_drift, m, p, W, ldt);
  __syncthreads();
  minv_mid(Ms, ld, sc + s, my, stn_drift, m, method, p, W, ldt, vgs[s],
           min_vg_val);
  __syncthreads();
  if (p > 0) minv_fin(Ms, ld, n, p, W, ldt);
}

int minv_steps(hipStream_t st, const double *Li, int64_t ld, int64_t stride,
               StepSc *sc, const int32_t *idx, int64_t N,
               const double *stn_drift, int m, int method, double *M,
               double *T0, const spk_vg *vgs, double min_vg_val, int S) {
  const int64_t nb = ceil_div(N, 64);
  const int p = method == SPK_M_SK ? 0 : method == SPK_M_EDK ? 1 + m : 1;
  if (N <= 64) {
    hipLaunchKernelGGL(k_minv_small, dim3(1, S), dim3(256), 0, st, Li, ld,
                       stride, sc, idx, N, stn_drift, m, method, p, M, T0, ld,
                       vgs, min_vg_val);
    return check_launch("k_minv");
  }
  hipLaunchKernelGGL(k_minv_tiles, dim3((unsigned)(nb * (nb + 1) / 2), S),
                     dim3(256), 0, st, Li, ld, stride, (const StepSc *)sc, M);
  if (p > 0)
    hipLaunchKernelGGL(k_minv_w, dim3((unsigned)nb, S), dim3(256), 0, st,
                       (const double *)M, ld, stride, (const StepSc *)sc, idx,
                       N, stn_drift, m, p, T0, ld);
  hipLaunchKernelGGL(k_minv_mid, dim3(S), dim3(256), 0, st, M, ld, stride, sc,
                     idx, N, stn_drift, m, method, p, T0, ld, vgs, min_vg_val);
  if (p > 0)
    hipLaunchKernelGGL(k_minv_fin,
                       dim3((unsigned)std::min<int64_t>(N, 256), S), dim3(256),
                       0, st, M, ld, stride, (const StepSc *)sc, p,
                       (const double *)T0, ld);
  return check_launch("k_minv");
}

// Li as float (column-major) for the FP32 contraction.
__global__ void k_cast_tri(const double *__restrict__ Li, float *__restrict__ L32,
                           int64_t ld, int64_t stride,
                           const StepSc *__restrict__ sc) {
  const int s = blockIdx.y;
  // only the steps of the FP32 contraction read L32
  if (sc[s].status || (sc[s].flags & (SPK_ST_FP64VAR | SPK_ST_INT8VAR)))
    return;
  const int n = sc[s].n;
  const int64_t tot = (int64_t)n * n;
  const double *src = Li + (int64_t)s * stride;
  float *dst = L32 + (int64_t)s * stride;
  for (int64_t e = blockIdx.x * 256 + threadIdx.x; e < tot;
       e += (int64_t)gridDim.x * 256) {
    const int i = (int)(e % n), j = (int)(e / n);
    dst[i + (int64_t)j * ld] = (float)src[i + (int64_t)j * ld];
  }
}

}  // namespace spk
