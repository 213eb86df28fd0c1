// Learned variogram proposal: synthetic Gaussian fields, variogram features
// and a small multilayer perceptron trained and run on the GPU.
//
//  spk_simulate_fields_dev : unconditional Gaussian fields at each step's
//                            active stations, z = mean + L xi with C = L L^T
//                            the step variogram's covariance (nugget on the
//                            diagonal), using the kriging kernels' assembly
//                            and Cholesky
//  spk_vg_features_dev     : 20 equal-width lag bins over (0, mdr * max
//                            distance]: semivariance / variance and the
//                            share of pairs per bin times the bin count
//                            (1 = uniform), 40 features
//  spk_mlp_*               : 40 -> 128 -> 128 -> 128 -> 6 with GELU;
//                            outputs = 3 model logits (Sph, Exp, Gau) and
//                            3 regressions (log sill/var, log range/max
//                            distance, nugget fraction); softmax cross-
//                            entropy + weighted squared error; Adam.
#include "spk_krige.h"

namespace spk {

// ---- synthetic fields ------------------------------------------------------
__global__ void k_sim_diag(double *__restrict__ A, int64_t ld, int64_t stride,
                           const StepSc *__restrict__ sc,
                           const spk_vg *__restrict__ vgs) {
  const int s = blockIdx.y;
  if (sc[s].status) return;
  const int n = sc[s].n;
  const spk_vg &vg = vgs[s];
  double nug = 0.0, tot = 0.0;
  for (int k = 0; k < vg.n; ++k) {
    tot += vg.sill[k];
    if (vg.type[k] == SPK_VG_NUG) nug += vg.sill[k];
  }
  double *As = A + (int64_t)s * stride;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    As[i + (int64_t)i * ld] += nug + 1e-6 * tot;
}

__device__ inline unsigned long long smix(unsigned long long x) {
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}

// standard normal from a counter (Box-Muller on two hashed uniforms)
__device__ inline double normal_at(unsigned long long seed,
                                   unsigned long long k) {
  const unsigned long long a = smix(seed ^ smix(2 * k));
  const unsigned long long b = smix(seed ^ smix(2 * k + 1));
  const double u1 = ((double)(a >> 11) + 0.5) * (1.0 / 9007199254740992.0);
  const double u2 = (double)(b >> 11) * (1.0 / 9007199254740992.0);
  return sqrt(-2.0 * log(u1)) * cos(2.0 * kPi * u2);
}

// z_i = mean + sum_{k <= i} L_ik xi_k at active station i, NaN elsewhere
__global__ __launch_bounds__(256) void k_sim_apply(
    const double *__restrict__ L, int64_t ld, int64_t stride,
    const StepSc *__restrict__ sc, const int32_t *__restrict__ idx,
    int64_t N, const double *__restrict__ means, unsigned long long seed,
    int64_t t0, double *__restrict__ out) {
  const int s = blockIdx.x;
  double *o = out + (int64_t)s * N;
  for (int64_t i = threadIdx.x; i < N; i += 256) o[i] = NAN;
  __syncthreads();
  if (sc[s].status) return;
  const int n = sc[s].n;
  const double *Ls = L + (int64_t)s * stride;
  const int32_t *my = idx + (int64_t)s * N;
  __shared__ double xi[256];
  const unsigned long long sd = smix(seed ^ smix((unsigned long long)(t0 + s)));
  for (int i0 = 0; i0 < n; i0 += 256) {
    double acc = 0.0;
    const int i = i0 + threadIdx.x;
    for (int k0 = 0; k0 <= i0; k0 += 256) {
      __syncthreads();
      xi[threadIdx.x] =
          (k0 + (int)threadIdx.x < n) ? normal_at(sd, k0 + threadIdx.x)
                                      : 0.0;
      __syncthreads();
      if (i < n) {
        const int kmax = min(256, i - k0 + 1);
        for (int k = 0; k < kmax; ++k)
          acc += Ls[i + (int64_t)(k0 + k) * ld] * xi[k];
      }
    }
    if (i < n) o[my[i]] = means[t0 + s] + acc;
  }
}

// ---- lag-bin features ---------------------------------------------------------
__global__ __launch_bounds__(256) void k_features(
    const int32_t *__restrict__ pi, const int32_t *__restrict__ pj,
    const double *__restrict__ pd, int64_t M, const double *__restrict__ vals,
    int64_t N, double mdr, int nlag, float *__restrict__ feat,
    double *__restrict__ scale) {
  const int s = blockIdx.x;
  const double *z = vals + (int64_t)s * N;
  const int tid = threadIdx.x;
  __shared__ double red[256];
  __shared__ double sums[64];
  __shared__ unsigned long long cnts[64];
  __shared__ double maxd_s, var_s;
  // mean and variance of the step's values
  double a = 0.0, c = 0.0;
  for (int64_t i = tid; i < N; i += 256)
    if (!isnan(z[i])) {
      a += z[i];
      c += 1.0;
    }
  red[tid] = a;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) red[tid] += red[tid + w];
    __syncthreads();
  }
  const double sa = red[0];
  __syncthreads();
  red[tid] = c;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) red[tid] += red[tid + w];
    __syncthreads();
  }
  const double sc = red[0];
  __syncthreads();
  const double mean = sa / sc;
  double v = 0.0;
  for (int64_t i = tid; i < N; i += 256)
    if (!isnan(z[i])) v += (z[i] - mean) * (z[i] - mean);
  red[tid] = v;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) red[tid] += red[tid + w];
    __syncthreads();
  }
  if (tid == 0) {
    var_s = red[0] / sc;
    // largest active pair distance: scan the sorted pairs from the end
    double md = 0.0;
    for (int64_t e = M - 1; e >= 0; --e)
      if (!isnan(z[pi[e]]) && !isnan(z[pj[e]])) {
        md = pd[e];
        break;
      }
    maxd_s = md * mdr;
    scale[2 * s] = maxd_s;
    scale[2 * s + 1] = var_s;
  }
  if (tid < 64) {
    sums[tid] = 0.0;
    cnts[tid] = 0;
  }
  __syncthreads();
  const double md = maxd_s;
  for (int64_t e = tid; md > 0.0 && e < M; e += 256) {
    const double d = pd[e];
    if (d > md) break;  // sorted: nothing beyond
    const double zi = z[pi[e]], zj = z[pj[e]];
    if (isnan(zi) || isnan(zj)) continue;
    int b = (int)(d / md * nlag);
    if (b >= nlag) b = nlag - 1;
    atomicAdd(&sums[b], 0.5 * (zi - zj) * (zi - zj));
    atomicAdd(&cnts[b], 1ull);
  }
  __syncthreads();
  if (tid == 0) {
    unsigned long long tot = 0;
    for (int b = 0; b < nlag; ++b) tot += cnts[b];
    float *f = feat + (int64_t)s * 2 * nlag;
    for (int b = 0; b < nlag; ++b) {
      const double g = cnts[b] ? sums[b] / cnts[b] : 0.0;
      f[b] = (float)(var_s > 0 ? g / var_s : 0.0);
      f[nlag + b] = (float)(tot ? (double)cnts[b] * nlag / tot : 0.0);
    }
  }
}

// ---- MLP -----------------------------------------------------------------------
// Layer sizes and the flat parameter layout [W1 b1 W2 b2 W3 b3 W4 b4] with
// W_l row-major [out x in].
constexpr int kIn = 40, kH = 128, kOut = 6, kNReg = 3, kNCls = 3;
__host__ __device__ constexpr int mlp_dim(int l) {
  return l == 0 ? kIn : (l == 4 ? kOut : kH);
}
__host__ __device__ constexpr int64_t w_off(int l) {  // l = 1..4
  int64_t o = 0;
  for (int k = 1; k < l; ++k) o += (int64_t)mlp_dim(k) * mlp_dim(k - 1) + mlp_dim(k);
  return o;
}
__host__ __device__ constexpr int64_t b_off(int l) {
  return w_off(l) + (int64_t)mlp_dim(l) * mlp_dim(l - 1);
}
constexpr int64_t kNParams = w_off(5);
constexpr int kMaxBatch = 1 << 21;

__device__ inline float gelu(float x) {
  return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f));
}
__device__ inline float gelu_d(float x) {
  const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
  return cdf + x * pdf;
}

typedef float mf4_t __attribute__((ext_vector_type(4)));
__device__ inline mf4_t mfma32(float a, float b, mf4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// four consecutive floats at any float's alignment
struct __attribute__((packed, aligned(4))) F4 {
  float v[4];
};

// Forward pass of 16 samples per workgroup through all layers on FP32 MFMA,
// activations in LDS; with TRAIN also the loss, its gradient with respect to
// the outputs and the backward pass to every layer's dZ:
// L = CE(softmax(y[0:3]), cls) + reg_w * sum_k (y[3+k] - t[k])^2 * m[k]
// where m masks regression targets that are NaN; a class outside 0..2 drops
// the cross-entropy term of that sample.  The weights (150 KB) come from L2.
// A layer's product runs k = kb + 4 lg + j for MFMA j of a group of 16, so
// that a lane reads four consecutive weights.  One launch in place of 8
// (forward) or 16 (with the backward pass): those were bound by their
// launches and, at 256 samples, by 16 to 64 workgroups each (about 110 us
// with the backward pass, now 25).
// hbuf: H_1 .. H_3 [B x 128] each; dbuf: dZ_1 .. dZ_3 [B x 128], dZ_4 [B x 6];
// lossp: one partial sum per workgroup.
template <bool TRAIN>
__global__ __launch_bounds__(256) void k_mlp(
    const float *__restrict__ P, const float *__restrict__ X, int B,
    float *__restrict__ out, const int32_t *__restrict__ cls,
    const float *__restrict__ tgt, float reg_w, float *__restrict__ hbuf,
    float *__restrict__ dbuf, float *__restrict__ lossp) {
  constexpr int LD = kH + 4;
  __shared__ __align__(16) float Hs[2][16][LD];  // layer in / out, dZ in / out
  __shared__ float Zs[3][16][LD];                // Z_1 .. Z_3
  __shared__ float lsum[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int r0 = blockIdx.x * 16;
  for (int e = tid; e < 16 * 48; e += 256) {
    const int i = e / 48, k = e % 48;
    Hs[0][i][k] = r0 + i < B && k < kIn ? X[(int64_t)(r0 + i) * kIn + k] : 0.f;
  }
  __syncthreads();
#pragma unroll
  for (int l = 1; l <= 4; ++l) {
    const int I = mlp_dim(l - 1), O = mlp_dim(l);
    const float *W = P + w_off(l), *bias = P + b_off(l);
    const float (*in)[LD] = Hs[(l - 1) & 1];
    float (*ou)[LD] = Hs[l & 1];
    for (int t = wave; t < (O + 15) / 16; t += 4) {
      const int col = t * 16 + li;
      mf4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < I; kb += 16) {
        const int k = kb + 4 * lg;
        F4 w = {{0.f, 0.f, 0.f, 0.f}};
        if (col < O && k < I)
          w = *reinterpret_cast<const F4 *>(W + (int64_t)col * I + k);
        const float4 h = *reinterpret_cast<const float4 *>(&in[li][k]);
        acc = mfma32(h.x, w.v[0], acc);
        acc = mfma32(h.y, w.v[1], acc);
        acc = mfma32(h.z, w.v[2], acc);
        acc = mfma32(h.w, w.v[3], acc);
      }
      if (col < O) {
        const float bc = bias[col];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 4 * lg + r;
          const float z = acc[r] + bc;
          if (l < 4) {
            const float h = gelu(z);
            ou[row][col] = h;
            if (TRAIN) {
              Zs[l - 1][row][col] = z;
              if (r0 + row < B)
                hbuf[((int64_t)(l - 1) * B + r0 + row) * kH + col] = h;
            }
          } else {
            ou[row][col] = z;
            if (!TRAIN && r0 + row < B)
              out[(int64_t)(r0 + row) * kOut + col] = z;
          }
        }
      }
    }
    __syncthreads();
  }
  if (!TRAIN) return;
  // the outputs are in Hs[0]; dZ_4 goes to Hs[1], zero beyond its 6 columns
  // (to the group of 16) and beyond the batch
  {
    const int i = tid >> 4, k = tid & 15;
    Hs[1][i][k] = 0.f;
  }
  __syncthreads();
  if (tid < 16) {
    float acc = 0.f;
    const int b = r0 + tid;
    if (b < B) {
      const float *y = Hs[0][tid];
      float *g = Hs[1][tid];
      const float mx = fmaxf(fmaxf(y[0], y[1]), y[2]);
      const float e0 = expf(y[0] - mx), e1 = expf(y[1] - mx),
                  e2 = expf(y[2] - mx);
      const float se = e0 + e1 + e2;
      const int c = cls[b];
      const float p[3] = {e0 / se, e1 / se, e2 / se};
      const bool has_c = c >= 0 && c < kNCls;  // other labels: no class term
      if (has_c) acc += -(y[c] - mx - logf(se));
      for (int k = 0; k < kNCls; ++k)
        g[k] = has_c ? (p[k] - (k == c ? 1.f : 0.f)) / B : 0.f;
      for (int k = 0; k < kNReg; ++k) {
        const float t = tgt[(int64_t)b * kNReg + k];
        if (isnan(t)) {
          g[kNCls + k] = 0.f;
          continue;
        }
        const float r = y[kNCls + k] - t;
        acc += reg_w * r * r;
        g[kNCls + k] = 2.f * reg_w * r / B;
      }
      for (int k = 0; k < kOut; ++k)
        dbuf[(int64_t)3 * B * kH + (int64_t)b * kOut + k] = g[k];
    }
    lsum[tid] = acc;
  }
  __syncthreads();
  if (tid == 0) {
    float acc = 0.f;
    for (int i = 0; i < 16; ++i) acc += lsum[i];
    lossp[blockIdx.x] = acc;
  }
  // dZ_{l-1} = (dZ_l W_l) * gelu'(Z_{l-1})
#pragma unroll
  for (int l = 4; l >= 2; --l) {
    const int O = mlp_dim(l);
    const float *W = P + w_off(l);
    const float (*in)[LD] = Hs[(l - 1) & 1];
    float (*ou)[LD] = Hs[l & 1];
    for (int t = wave; t < kH / 16; t += 4) {
      const int col = t * 16 + li;
      mf4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
      for (int kb = 0; kb < O; kb += 16) {
        const int k = kb + 4 * lg;
        float w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          w[j] = k + j < O ? W[(int64_t)(k + j) * kH + col] : 0.f;
        const float4 d = *reinterpret_cast<const float4 *>(&in[li][k]);
        acc = mfma32(d.x, w[0], acc);
        acc = mfma32(d.y, w[1], acc);
        acc = mfma32(d.z, w[2], acc);
        acc = mfma32(d.w, w[3], acc);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * lg + r;
        const float d = acc[r] * gelu_d(Zs[l - 2][row][col]);
        ou[row][col] = d;
        if (r0 + row < B)
          dbuf[((int64_t)(l - 2) * B + r0 + row) * kH + col] = d;
      }
    }
    __syncthreads();
  }
}

// Weight and bias gradients dW_l = dZ_l^T H_{l-1}, db_l = sum dZ_l of all
// layers: one 16 x 16 tile per workgroup (kGradTiles over the layers), its
// batch rows [blockIdx.y * rows, ...) dealt to the four waves, whose sums are
// added in wave order.  part: the gradients themselves (one row chunk) or one
// copy per chunk for k_grad_sum.  The first workgroup also sums the loss.
// (Four products, each with 8 to 64 workgroups that walked all rows, and four
// bias sums with one thread per output took 250 us at 256 samples, this 7.5.)
constexpr int kGradTiles = 8 * 3 + 8 * 8 + 8 * 8 + 8;
__global__ __launch_bounds__(256) void k_mlp_grad(
    const float *__restrict__ X, int B, const float *__restrict__ hbuf,
    const float *__restrict__ dbuf, int rows, float *__restrict__ part,
    const float *__restrict__ lossp, int nloss, float *__restrict__ loss) {
  __shared__ float red[4][17][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lg = lane >> 4;
  int t = blockIdx.x, l = 1;
  if (t < 24) {
    l = 1;
  } else if ((t -= 24) < 64) {
    l = 2;
  } else if ((t -= 64) < 64) {
    l = 3;
  } else {
    t -= 64;
    l = 4;
  }
  const int I = mlp_dim(l - 1), O = mlp_dim(l);
  const int nti = (I + 15) / 16;
  const int o = (t / nti) * 16 + li, i = (t % nti) * 16 + li;
  const float *dZ = dbuf + (int64_t)(l - 1) * B * kH;
  const float *H = l == 1 ? X : hbuf + (int64_t)(l - 2) * B * kH;
  const int b0 = blockIdx.y * rows, b1 = min(B, b0 + rows);
  mf4_t acc = {0.f, 0.f, 0.f, 0.f};
  float db = 0.f;
#pragma unroll 4
  for (int b = b0 + 4 * wave + lg; b - lg < b1; b += 16) {
    const bool in = b < b1;
    const float d = in && o < O ? dZ[(int64_t)b * O + o] : 0.f;
    const float h = in && i < I ? H[(int64_t)b * I + i] : 0.f;
    db += d;
    acc = mfma32(d, h, acc);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][4 * lg + r][li] = acc[r];
  db += __shfl_xor(db, 16, 64);
  db += __shfl_xor(db, 32, 64);
  if (lg == 0) red[wave][16][li] = db;
  __syncthreads();
  float *g = part + (int64_t)blockIdx.y * kNParams;
  {
    const int r = tid >> 4, c = tid & 15;
    const int oo = (t / nti) * 16 + r, ii = (t % nti) * 16 + c;
    if (oo < O && ii < I)
      g[w_off(l) + (int64_t)oo * I + ii] =
          red[0][r][c] + red[1][r][c] + red[2][r][c] + red[3][r][c];
  }
  if (t % nti == 0 && tid < 16 && o < O)
    g[b_off(l) + o] =
        red[0][16][li] + red[1][16][li] + red[2][16][li] + red[3][16][li];
  if (blockIdx.x || blockIdx.y) return;
  __shared__ float ls[256];
  float v = 0.f;
  for (int e = tid; e < nloss; e += 256) v += lossp[e];
  ls[tid] = v;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) ls[tid] += ls[tid + w];
    __syncthreads();
  }
  if (tid == 0) loss[0] = ls[0] / B;
}

__global__ __launch_bounds__(256) void k_grad_sum(
    const float *__restrict__ part, int n, float *__restrict__ grads) {
  const int64_t e = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (e >= kNParams) return;
  float v = 0.f;
  for (int k = 0; k < n; ++k) v += part[k * kNParams + e];
  grads[e] = v;
}

__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g,
                       float *__restrict__ m, float *__restrict__ v,
                       int64_t n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  for (int64_t e = blockIdx.x * 256 + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * 256) {
    const float gi = g[e];
    const float mi = b1 * m[e] + (1.f - b1) * gi;
    const float vi = b2 * v[e] + (1.f - b2) * gi * gi;
    m[e] = mi;
    v[e] = vi;
    p[e] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

__global__ void k_init_params(float *__restrict__ p, unsigned long long seed) {
  for (int64_t e = blockIdx.x * 256 + threadIdx.x; e < kNParams;
       e += (int64_t)gridDim.x * 256) {
    int l = 1;
    while (l < 4 && e >= w_off(l + 1)) ++l;
    const bool is_w = e < b_off(l);
    const double u =
        (double)(smix(seed ^ smix((unsigned long long)e)) >> 11) *
        (1.0 / 9007199254740992.0);
    // uniform(-1/sqrt(in), 1/sqrt(in)) for weights and biases
    const float lim = 1.0f / sqrtf((float)mlp_dim(l - 1));
    p[e] = (float)((2.0 * u - 1.0) * lim) * (is_w ? 1.0f : 0.5f);
  }
}

}  // namespace spk

using namespace spk;

extern "C" {

int spk_simulate_fields_dev(spk_ctx *ctx, const spk_problem *prob, int64_t T,
                            const double *mask_vals, const spk_vg *vgs,
                            const double *means, uint64_t seed, double *out,
                            int32_t *info) {
  if (!ctx || !prob || !mask_vals || !vgs || !means || !out || !info)
    return set_error(SPK_EARG, "null argument");
  const int64_t N = prob->n_stns;
  if (N < 2) return set_error(SPK_ESHAPE, "need stations");
  if (ctx->pairs_sorted)
    return set_error(SPK_EARG,
                     "field simulation after a station-pair sort on the same "
                     "context is disabled (that order has not been run since "
                     "a lock that stalled it was mended): simulate first, or "
                     "use another context");
  if (T <= 0) return SPK_OK;
  SPK_HIP(hipSetDevice(ctx->device));
  hipStream_t sm = ctx->stream;
  double *sx;
  SPK_TRY(ws_get(ctx, "stn_xy", 2 * N * sizeof(double), (void **)&sx));
  double *sy = sx + N;
  SPK_TRY(recenter(sm, prob, sx, sy, nullptr, nullptr));
  const int64_t ld = ((N + 63) / 64) * 64;
  const int64_t strideM = ld * ld;
  const int64_t ldz = ld;
  const int64_t S = std::max<int64_t>(1, std::min<int64_t>(
      64, (int64_t)((size_t)4 << 30) / (strideM * 8)));
  int32_t *idx;
  double *zact, *A;
  StepSc *sc;
  SPK_TRY(ws_get(ctx, "sim_idx", S * N * 4, (void **)&idx));
  SPK_TRY(ws_get(ctx, "sim_z", S * ldz * 8, (void **)&zact));
  SPK_TRY(ws_get(ctx, "sim_sc", S * sizeof(StepSc), (void **)&sc));
  SPK_TRY(ws_get(ctx, "sim_A", S * strideM * 8, (void **)&A));
  const int tiles = (int)ceil_div(N, 64);
  for (int64_t t0 = 0; t0 < T; t0 += S) {
    const int Sb = (int)std::min<int64_t>(S, T - t0);
    hipLaunchKernelGGL(k_compact, dim3(Sb), dim3(256), 0, sm,
                       mask_vals + t0 * N, N, idx, zact, ldz, sc,
                       (const spk_vg *)nullptr, SPK_M_NNB, -INFINITY, 0.0,
                       (const int32_t *)nullptr);
    hipLaunchKernelGGL(k_assemble, dim3(tiles * tiles, Sb), dim3(256), 0, sm,
                       sx, sy, idx, N, sc, vgs + t0, 1, -INFINITY, A, ld,
                       strideM, (double *)nullptr);
    hipLaunchKernelGGL(k_sim_diag, dim3(8, Sb), dim3(256), 0, sm, A, ld,
                       strideM, sc, vgs + t0);
    SPK_TRY(chol_steps(sm, A, ld, strideM, sc, vgs + t0, 0, N, Sb));
    hipLaunchKernelGGL(k_sim_apply, dim3(Sb), dim3(256), 0, sm, A, ld, strideM,
                       sc, idx, N, means, (unsigned long long)seed, t0,
                       out + t0 * N);
    hipLaunchKernelGGL(k_status_out, dim3((unsigned)ceil_div(Sb, 256)),
                       dim3(256), 0, sm, sc, Sb, info + t0, (double *)nullptr);
    SPK_TRY(check_launch("simulate"));
  }
  return SPK_OK;
}

int spk_vg_features_dev(spk_ctx *ctx, const int32_t *pi, const int32_t *pj,
                        const double *pd, int64_t M, int64_t N,
                        const double *vals, int64_t T, double mdr, int nlag,
                        float *feat, double *scale) {
  if (!ctx || !pi || !pj || !pd || !vals || !feat || !scale)
    return set_error(SPK_EARG, "null argument");
  if (nlag < 1 || nlag > 64) return set_error(SPK_EARG, "nlag in 1..64");
  if (T <= 0) return SPK_OK;
  SPK_HIP(hipSetDevice(ctx->device));
  for (int64_t t0 = 0; t0 < T; t0 += 65535) {
    const int Tb = (int)std::min<int64_t>(65535, T - t0);
    hipLaunchKernelGGL(k_features, dim3(Tb), dim3(256), 0, ctx->stream, pi, pj,
                       pd, M, vals + t0 * N, N, mdr, nlag,
                       feat + t0 * 2 * nlag, scale + t0 * 2);
    SPK_TRY(check_launch("k_features"));
  }
  return SPK_OK;
}

int64_t spk_mlp_n_params(void) { return kNParams; }

int spk_mlp_init_dev(spk_ctx *ctx, uint64_t seed, float *params) {
  if (!ctx || !params) return set_error(SPK_EARG, "null argument");
  SPK_HIP(hipSetDevice(ctx->device));
  hipLaunchKernelGGL(k_init_params, dim3(64), dim3(256), 0, ctx->stream,
                     params, (unsigned long long)seed);
  return check_launch("k_init_params");
}

int spk_mlp_forward_dev(spk_ctx *ctx, const float *params, const float *X,
                        int B, float *out) {
  if (!ctx || !params || !X || !out) return set_error(SPK_EARG, "null argument");
  if (B <= 0) return SPK_OK;
  if (B > kMaxBatch) return set_error(SPK_ESHAPE, "batch above %d", kMaxBatch);
  SPK_HIP(hipSetDevice(ctx->device));
  hipLaunchKernelGGL((k_mlp<false>), dim3((unsigned)ceil_div(B, 16)),
                     dim3(256), 0, ctx->stream, params, X, B, out,
                     (const int32_t *)nullptr, (const float *)nullptr, 0.f,
                     (float *)nullptr, (float *)nullptr, (float *)nullptr);
  return check_launch("k_mlp");
}

int spk_mlp_loss_grad_dev(spk_ctx *ctx, const float *params, const float *X,
                          int B, const int32_t *cls, const float *reg,
                          float reg_w, float *grads, float *loss) {
  if (!ctx || !params || !X || !cls || !reg || !grads || !loss)
    return set_error(SPK_EARG, "null argument");
  if (B <= 0) return set_error(SPK_EARG, "empty batch");
  if (B > kMaxBatch) return set_error(SPK_ESHAPE, "batch above %d", kMaxBatch);
  SPK_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  const int nblk = (int)ceil_div(B, 16);
  // row chunks of at least 256 samples, at most 32 of them
  const int nch = (int)std::min<int64_t>(32, ceil_div(B, 256));
  const int rows = (int)ceil_div(ceil_div(B, nch), 16) * 16;
  float *hbuf, *dbuf, *lossp, *part = grads;
  SPK_TRY(ws_get(ctx, "mlp_h", 3 * (int64_t)B * kH * 4, (void **)&hbuf));
  SPK_TRY(ws_get(ctx, "mlp_d", (int64_t)B * (3 * kH + kOut) * 4,
                 (void **)&dbuf));
  SPK_TRY(ws_get(ctx, "mlp_loss", (int64_t)nblk * 4, (void **)&lossp));
  if (nch > 1)
    SPK_TRY(ws_get(ctx, "mlp_part", nch * kNParams * 4, (void **)&part));
  hipLaunchKernelGGL((k_mlp<true>), dim3((unsigned)nblk), dim3(256), 0, st,
                     params, X, B, (float *)nullptr, cls, reg, reg_w, hbuf,
                     dbuf, lossp);
  hipLaunchKernelGGL(k_mlp_grad, dim3(kGradTiles, (unsigned)nch), dim3(256), 0,
                     st, X, B, (const float *)hbuf, (const float *)dbuf, rows,
                     part, (const float *)lossp, nblk, loss);
  if (nch > 1)
    hipLaunchKernelGGL(k_grad_sum, dim3((unsigned)ceil_div(kNParams, 256)),
                       dim3(256), 0, st, (const float *)part, nch, grads);
  return check_launch("k_mlp_grad");
}

int spk_mlp_adam_dev(spk_ctx *ctx, float *params, const float *grads,
                     float *m, float *v, int64_t step, float lr, float b1,
                     float b2, float eps) {
  if (!ctx || !params || !grads || !m || !v)
    return set_error(SPK_EARG, "null argument");
  if (step < 1) return set_error(SPK_EARG, "step counts from 1");
  SPK_HIP(hipSetDevice(ctx->device));
  const float c1 = 1.f - powf(b1, (float)step);
  const float c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_adam, dim3(64), dim3(256), 0, ctx->stream, params,
                     grads, m, v, kNParams, lr, b1, b2, eps, c1, c2);
  return check_launch("k_adam");
}

}  // extern "C"
