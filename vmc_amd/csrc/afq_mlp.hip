// Learned exchange-energy surrogate: a GELU MLP F -> H -> H -> H -> 1 with
// FP32 master weights, every GEMM on BF16 MFMA (operands rounded to bf16 when
// staged in LDS) with FP32 accumulation, trained with MSE + Adam on the GPU.
//
// Input (per walker): Re fb_g (g < G) and Re diag G_s (two spins, N each),
// standardised with the training set's mean / std.  Target: the exchange energy
// E_K = 1/2 sum_s m_s sum_g tr(f_{s,g} f_{s,g}) relative to the Coulomb energy
// E_J = 1/2 sum_g fb_g^2 that is computed exactly anyway: y = E_K - E_J.  The two
// are strongly correlated and largely cancel in E_L, so y has a much smaller
// spread than E_K.
#include <math.h>

#include <algorithm>
#include <stdexcept>
#include <string>

#include <hipcub/hipcub.hpp>

#include "afq_device.hpp"
#include "afq_internal.hpp"

namespace afq {

static inline unsigned cdivu(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_d(float z) {
  return 0.5f * (1.f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// ---------------------------------------------------------------- GEMM (bf16 operands, fp32 accumulate)
// workgroup z takes k in [z kc, (z + 1) kc); with part it stores its FP32 sum to part[z][r][c]
template <bool A_ROWFAST, class LA, class LB, class EP>
__global__ __launch_bounds__(256) void k_gemm_bf16e(LA la, LB lb, EP ep, int M, int N, int K, int kc, float* part) {
  using Eng = MmaBF16E<64, 64, 2, 2, A_ROWFAST>;
  __shared__ __attribute__((aligned(16))) u16 lds[Eng::LDS_BYTES / 2];
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64, k0 = blockIdx.z * kc, kn = min(kc, K - k0);
  Eng e;
  // (no branch around a load: an element outside reads a valid one and is replaced by zero,
  // so that all loads of a stage are in flight together)
  e.run([&](int r, int k) {
          const float v = la(min(r0 + r, M - 1), k0 + min(k, kn - 1));
          return r0 + r < M && k < kn ? v : 0.f;
        },
        [&](int k, int c) {
          const float v = lb(k0 + min(k, kn - 1), min(c0 + c, N - 1));
          return k < kn && c0 + c < N ? v : 0.f;
        },
        kn, lds);
  float* o = part + (int64_t)blockIdx.z * M * N;
  e.store([&](int r, int c, float v) {
    if (r0 + r < M && c0 + c < N) {
      if (part) o[(int64_t)(r0 + r) * N + c0 + c] = v;
      else ep(r0 + r, c0 + c, v);
    }
  });
}
// out[e] = sum of the nz partial sums of element e, in order
__global__ __launch_bounds__(256) void k_sum_parts(const float* __restrict__ part, float* __restrict__ out, int64_t n, int nz) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= n) return;
  float s = 0.f;
  for (int z = 0; z < nz; ++z) s += part[(int64_t)z * n + e];
  out[e] = s;
}
template <bool A_ROWFAST = false, class LA, class LB, class EP>
static void gemm(const LA& la, const LB& lb, const EP& ep, int M, int N, int K, hipStream_t st) {
  hipLaunchKernelGGL((k_gemm_bf16e<A_ROWFAST, LA, LB, EP>), dim3(cdivu(N, 64), cdivu(M, 64)), dim3(256), 0, st, la, lb, ep, M,
                     N, K, K, (float*)nullptr);
}
// Weight gradients: a small output (M x N) summed over the batch.  One workgroup per output
// tile left 16 of them (256 x 256) walking a batch of 4096 (0.50 ms; 0.84 ms for the 40 of
// 600 x 256); with the batch in chunks of at least 128 over up to 1024 workgroups, the FP32
// partial sums added in order (9 us), rows loaded coalesced and all loads of a stage in
// flight together: 13 to 30 us.
static int wgrad_chunks(int M, int N, int B) {
  const int tiles = (int)(cdivu(M, 64) * cdivu(N, 64));
  return (int)std::max(1u, std::min(cdivu(1024, tiles), (unsigned)(B / 128)));
}
int64_t mlp_ws_floats(const int* dims, int B) {
  int64_t most = 0;
  for (int l = 0; l < 4; ++l)
    most = std::max(most, (int64_t)wgrad_chunks(dims[l], dims[l + 1], B) * dims[l] * dims[l + 1]);
  return most;
}
template <class LA, class LB>
static void gemm_wgrad(const LA& la, const LB& lb, float* out, float* ws, int M, int N, int B, hipStream_t st);

// operand views
struct Rows {  // H[r][k], row length K
  const float* H; int K;
  __device__ float operator()(int r, int k) const { return H[(int64_t)r * K + k]; }
};
struct RowsT {  // (r, k) -> H[k][r]
  const float* H; int K;
  __device__ float operator()(int r, int k) const { return H[(int64_t)k * K + r]; }
};
struct WB {  // W[k][c] (in x out)
  const float* W; int N;
  __device__ float operator()(int k, int c) const { return W[(int64_t)k * N + c]; }
};
struct WBT {  // (o, i) -> W[i][o]
  const float* W; int N;
  __device__ float operator()(int k, int c) const { return W[(int64_t)c * N + k]; }
};
struct FwdEp {
  float* z; float* h; const float* bias; int N; int act;
  __device__ void operator()(int r, int c, float v) const {
    const float zz = v + bias[c];
    z[(int64_t)r * N + c] = zz;
    h[(int64_t)r * N + c] = act ? gelu(zz) : zz;
  }
};
struct StoreEp {
  float* out; int N;
  __device__ void operator()(int r, int c, float v) const { out[(int64_t)r * N + c] = v; }
};
template <class LA, class LB>
static void gemm_wgrad(const LA& la, const LB& lb, float* out, float* ws, int M, int N, int B, hipStream_t st) {
  const int want = wgrad_chunks(M, N, B), kc = (int)cdivu(cdivu(B, want), 32) * 32, nz = (int)cdivu(B, kc);
  if (nz == 1) {
    gemm<true>(la, lb, StoreEp{out, N}, M, N, B, st);
    return;
  }
  hipLaunchKernelGGL((k_gemm_bf16e<true, LA, LB, StoreEp>), dim3(cdivu(N, 64), cdivu(M, 64), nz), dim3(256), 0, st, la, lb,
                     StoreEp{out, N}, M, N, B, kc, ws);
  hipLaunchKernelGGL(k_sum_parts, dim3(cdivu((int64_t)M * N, 256)), dim3(256), 0, st, ws, out, (int64_t)M * N, nz);
}

// ---------------------------------------------------------------- small kernels
// xn[b][f] = (X[idx[b]][f] - mu[f]) / sd[f]: the standardised input rows of a batch
__global__ __launch_bounds__(256) void k_standardize(const float* __restrict__ X, const int* __restrict__ idx,
                                                     const float* __restrict__ mu, const float* __restrict__ sd,
                                                     float* __restrict__ xn, int B, int F) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (int64_t)B * F) return;
  const int b = (int)(e / F), f = (int)(e - (int64_t)b * F), row = idx ? idx[b] : b;
  xn[e] = (X[(int64_t)row * F + f] - mu[f]) / sd[f];
}
// dz[i] = dh[i] gelu'(z[i]), in place: the weight and the input gradient and the bias
// gradient read it, which would each evaluate gelu' again for every tile they load
__global__ __launch_bounds__(256) void k_dz(float* __restrict__ dh, const float* __restrict__ z, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dh[i] *= gelu_d(z[i]);
}
// db[c] = sum_b dz[b][c]: a workgroup per 16 columns, 64 threads a column, then a tree (one
// thread a column over a batch of 4096 took 1.36 ms, this takes 0.019)
__global__ __launch_bounds__(1024) void k_colsum(const float* __restrict__ dz, float* __restrict__ db, int B, int N) {
  __shared__ float red[64][17];
  const int cc = threadIdx.x & 15, g = threadIdx.x >> 4, c = blockIdx.x * 16 + cc;
  float s = 0.f;
  if (c < N)
    for (int b = g; b < B; b += 64) s += dz[(int64_t)b * N + c];
  red[g][cc] = s;
  for (int o = 32; o > 0; o >>= 1) {
    __syncthreads();
    if (g < o) red[g][cc] += red[g + o][cc];
  }
  if (g == 0 && c < N) db[c] = red[0][cc];
}
// dy = (y - t_std)/B with t_std = (t - t_mu)/t_sd ; loss = 1/2 mean (y - t_std)^2
__global__ void k_loss(const float* y, const float* t, const int* idx, float* dy, float* lossp, int B, float tmu,
                       float tsd) {
  __shared__ float red[256];
  float l = 0.f;
  for (int b = threadIdx.x; b < B; b += blockDim.x) {
    const float ts = (t[idx ? idx[b] : b] - tmu) / tsd;
    const float d = y[b] - ts;
    dy[b] = d / B;
    l += 0.5f * d * d;
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) lossp[0] = red[0] / B;
}
__global__ void k_adam(float* p, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

// features of walkers idx[0..n): row j of X at dst0 + j
__global__ __launch_bounds__(256) void k_features(const double* fb, const double* theta, const double* phi0,
                                                  const double* phi1, const int* idx, float* X, int64_t dst0, int G,
                                                  int N, int64_t Ktot, Slot s0, Slot s1, int nslots, int F) {
  const int j = blockIdx.x;
  const int w = idx ? idx[j] : j;
  float* x = X + (dst0 + j) * F;
  for (int g = threadIdx.x; g < G; g += blockDim.x) x[g] = (float)fb[(int64_t)w * 2 * G + 2 * g];
  for (int e = threadIdx.x; e < 2 * N; e += blockDim.x) {
    const int sp = e / N, i = e - sp * N;
    const Slot sl = (sp == 0 || nslots == 1) ? s0 : s1;
    const double* ph = sl.phi == 0 ? phi0 : phi1;
    const double* th = theta + (int64_t)w * 2 * Ktot + 2 * sl.koff + (int64_t)i * 2 * sl.n;
    double d = 0.0;
    for (int q = 0; q < sl.n; ++q) d += th[2 * q] * ph[(int64_t)i * sl.n + q];
    x[G + e] = (float)d;
  }
}

// exact exchange energy E_K of walkers idx[0..n) from the exchange partials; yout
// (training target) receives E_K - E_J, E_J = 1/2 sum_{g<GE} Re fb_g^2
__global__ void k_ek(const double* Xp, const double* fb, const int* idx, const int* n_dev, int n, double* ek,
                     float* yout, int64_t dst0, int W, int nslots, int m0, int m1, int ngt0, int ngt1, int ngt_cap, int G,
                     int GE) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (n_dev) n = *n_dev;   // the grid covers the bound n was
  if (j >= n) return;
  const int w = idx ? idx[j] : j;
  double s = 0.0;
  for (int q = 0; q < nslots; ++q) {
    const int m = q == 0 ? m0 : m1, nt = q == 0 ? ngt0 : ngt1;
    for (int t = 0; t < nt; ++t) s += m * Xp[2 * (((int64_t)q * W + w) * ngt_cap + t)];
  }
  s *= 0.5;
  if (ek) ek[w] = s;
  if (yout) {
    double ej = 0.0;
    for (int g = 0; g < GE; ++g) {
      const double a = fb[(int64_t)w * 2 * G + 2 * g], b = fb[(int64_t)w * 2 * G + 2 * g + 1];
      ej += a * a - b * b;
    }
    yout[dst0 + j] = (float)(s - 0.5 * ej);
  }
}

// E_J = 1/2 sum_{g<GE} Re fb_g^2 of every walker (risk score of the control variate)
__global__ __launch_bounds__(64) void k_ej(const double* fb, double* ej, int G, int GE) {
  const int w = blockIdx.x, lane = threadIdx.x;
  double jr = 0.0;
  for (int g = lane; g < GE; g += 64) {
    const double a = fb[(int64_t)w * 2 * G + 2 * g], b = fb[(int64_t)w * 2 * G + 2 * g + 1];
    jr += a * a - b * b;
  }
  jr = wave_sum(jr);
  if (lane == 0) ej[w] = 0.5 * jr;
}

// control-variate local energy.  S_w - soff predicts y = E_K - E_J, so the
// surrogate energy is e_s = ecore + e1 - (S_w - soff) + delta and the exact one
// e_x = ecore + e1 - y + delta; both are clipped to center[w / nwr] -+ halfw (halfw > 0)
// as the population-control estimator clips every local energy.  soff is read from the
// device (*soff_dev), where the statistics of earlier measurements keep it.  A walker in the
// exact set (inclusion probability 1/pinv[w]) reports e_s + pinv[w] (e_x - e_s),
// an unbiased (Horvitz-Thompson) estimate of its clipped exact energy for any soff
// fixed before the exact set is drawn; dres[w] = e_x - e_s for the exact set.
__global__ __launch_bounds__(64) void k_energy_cv(const double* fb, const double* e1, const double* S,
                                                  const double* ek, const float* pinv,
                                                  const double* weights, double* eloc, double* dres, int G, int GE,
                                                  int nslots, int m0, int m1, double ecore, double delta,
                                                  const double* soff_dev, const double* center, int nwr, double halfw) {
  const int w = blockIdx.x, lane = threadIdx.x;
  const double soff = *soff_dev;
  double jr = 0.0;
  for (int g = lane; g < GE; g += 64) {
    const double a = fb[(int64_t)w * 2 * G + 2 * g], b = fb[(int64_t)w * 2 * G + 2 * g + 1];
    jr += a * a - b * b;
  }
  jr = wave_sum(jr);
  if (lane == 0) {
    const double lo = center && halfw > 0.0 ? center[w / nwr] - halfw : -INFINITY;
    const double hi = center && halfw > 0.0 ? center[w / nwr] + halfw : INFINITY;
    double base = ecore + delta;
    for (int s = 0; s < nslots; ++s) base += (s == 0 ? m0 : m1) * e1[2 * ((int64_t)w * nslots + s)];
    const double es = fmin(fmax(base - (S[w] - soff), lo), hi);
    double er = es, d = 0.0;
    if (pinv[w] > 0.f) {
      const double ex = fmin(fmax(base - (ek[w] - 0.5 * jr), lo), hi);
      d = ex - es;
      er += (double)pinv[w] * d;
    }
    const bool live = weights == nullptr || weights[w] != 0.0;
    eloc[w] = live ? er : 0.0;
    dres[w] = live ? d : 0.0;
  }
}

__global__ void k_pred_to_double(const float* y, double* S, int n, float tmu, float tsd) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) S[j] = (double)y[j] * tsd + tmu;
}

// ---------------------------------------------------------------- host side
static void hcheck(hipError_t e, const char* what) {
  if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

void mlp_forward(const Mlp& m, const float* X, const int* idx, int B, hipStream_t st) {
  const int* d = m.dims;
  hipLaunchKernelGGL(k_standardize, dim3(cdivu((int64_t)B * d[0], 256)), dim3(256), 0, st, X, idx, m.mu, m.sd, m.xn, B, d[0]);
  gemm(Rows{m.xn, d[0]}, WB{m.w[0], d[1]}, FwdEp{m.z[0], m.h[0], m.b[0], d[1], 1}, B, d[1], d[0], st);
  for (int l = 1; l < 4; ++l)
    gemm(Rows{m.h[l - 1], d[l]}, WB{m.w[l], d[l + 1]}, FwdEp{m.z[l], m.h[l], m.b[l], d[l + 1], l < 3 ? 1 : 0}, B,
         d[l + 1], d[l], st);
}

// gradients of 1/2 mean (y - t)^2 for the batch of the last mlp_forward (m.xn holds its input,
// m.h[3] y); dy already in m.dh[3]
void mlp_backward(const Mlp& m, int B, hipStream_t st) {
  const int* d = m.dims;
  for (int l = 3; l >= 0; --l) {
    const int64_t nz = (int64_t)B * d[l + 1];
    if (l < 3) hipLaunchKernelGGL(k_dz, dim3(cdivu(nz, 256)), dim3(256), 0, st, m.dh[l], m.z[l], nz);
    const Rows dz{m.dh[l], d[l + 1]};
    // dW_l = in_l^T dZ_l
    gemm_wgrad(RowsT{l ? m.h[l - 1] : m.xn, d[l]}, dz, m.gw[l], m.ws, d[l], d[l + 1], B, st);
    hipLaunchKernelGGL(k_colsum, dim3(cdivu(d[l + 1], 16)), dim3(1024), 0, st, m.dh[l], m.gb[l], B, d[l + 1]);
    // dH_{l-1} = dZ_l W_l^T
    if (l > 0) gemm(dz, WBT{m.w[l], d[l + 1]}, StoreEp{m.dh[l - 1], d[l]}, B, d[l], d[l + 1], st);
  }
}

float mlp_loss(const Mlp& m, const float* t, const int* idx, int B, hipStream_t st) {
  hipLaunchKernelGGL(k_loss, dim3(1), dim3(256), 0, st, m.h[3], t, idx, m.dh[3], m.lossbuf, B, m.t_mu, m.t_sd);
  float l = 0.f;
  hcheck(hipMemcpyAsync(&l, m.lossbuf, sizeof(float), hipMemcpyDeviceToHost, st), "loss D2H");
  hcheck(hipStreamSynchronize(st), "loss sync");
  return l;
}

void mlp_adam(Mlp& m, float lr, hipStream_t st) {
  m.t += 1;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - powf(b1, (float)m.t), c2 = 1.f - powf(b2, (float)m.t);
  for (int l = 0; l < 4; ++l) {
    const int64_t nw = (int64_t)m.dims[l] * m.dims[l + 1], nb = m.dims[l + 1];
    hipLaunchKernelGGL(k_adam, dim3(cdivu(nw, 256) > 1024 ? 1024 : cdivu(nw, 256)), dim3(256), 0, st, m.w[l], m.gw[l],
                       m.mw[l], m.vw[l], nw, lr, b1, b2, eps, c1, c2);
    hipLaunchKernelGGL(k_adam, dim3(cdivu(nb, 256)), dim3(256), 0, st, m.b[l], m.gb[l], m.mb[l], m.vb[l], nb, lr, b1,
                       b2, eps, c1, c2);
  }
}

void launch_features(const DevState& s, const int* idx, int n, float* X, int64_t dst0, hipStream_t st) {
  hipLaunchKernelGGL(k_features, dim3(n), dim3(256), 0, st, s.fb, s.theta, s.phi[0], s.phi[1], idx, X, dst0, s.G, s.N,
                     s.Ktot, s.slot[0], s.slot[s.nslots > 1 ? 1 : 0], s.nslots, s.G + 2 * s.N);
}

void launch_ek(const DevState& s, const int* idx, int n, double* ek, float* yout, int64_t dst0, hipStream_t st,
               const int* n_dev) {
  const int ng0 = (int)cdivu(s.GE, exchange_tile_g(s.slot[0].n));
  const int ng1 = s.nslots > 1 ? (int)cdivu(s.GE, exchange_tile_g(s.slot[1].n)) : 0;
  hipLaunchKernelGGL(k_ek, dim3(cdivu(n, 256)), dim3(256), 0, st, s.Xp, s.fb, idx, n_dev, n, ek, yout, dst0, s.W, s.nslots,
                     s.slot[0].mult, s.nslots > 1 ? s.slot[1].mult : 0, ng0, ng1, s.ngt_cap, s.G, s.GE);
}

__global__ void k_sub(double* a, const double* b, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] -= b[i];
}

void launch_sub(double* a, const double* b, int n, hipStream_t st) {
  hipLaunchKernelGGL(k_sub, dim3(cdivu(n, 256)), dim3(256), 0, st, a, b, n);
}

void launch_ej(const DevState& s, double* ej, hipStream_t st) {
  hipLaunchKernelGGL(k_ej, dim3(s.W), dim3(64), 0, st, s.fb, ej, s.G, s.GE);
}

void launch_predict(const DevState& s, const Mlp& m, const float* X, int n, double* S, hipStream_t st) {
  mlp_forward(m, X, nullptr, n, st);
  hipLaunchKernelGGL(k_pred_to_double, dim3(cdivu(n, 256)), dim3(256), 0, st, m.h[3], S, n, m.t_mu, m.t_sd);
  (void)s;
}

void launch_energy_cv(const DevState& s, const double* S, const double* ek, const float* pinv, double delta,
                      const double* soff_dev, const double* center, int nwr, double halfw, double* dres,
                      hipStream_t st) {
  hipLaunchKernelGGL(k_energy_cv, dim3(s.W), dim3(64), 0, st, s.fb, s.e1, S, ek, pinv, s.weights, s.eloc, dres, s.G,
                     s.GE, s.nslots, s.slot[0].mult, s.nslots > 1 ? s.slot[1].mult : 0, s.ecore, delta, soff_dev,
                     center, nwr, halfw);
}

// ---------------------------------------------------------------- exact set of the control variate
// One workgroup.  live[0 .. *nlive) lists the walkers of nonzero weight in ascending
// order; risky (nullable) flags the risk stratum.  sel receives the risk stratum
// (ascending) followed by one walker drawn uniformly from each consecutive block of m
// remaining live walkers (the last block may be shorter); pinv[w] is 1 for the risk
// stratum, the block's size for a drawn walker and 0 for every other walker, so that
// e_s + pinv (e_x - e_s) is an unbiased (Horvitz-Thompson) estimate of every walker's
// e_x.  The block draws are Philox(seed, (block, draw)) uniforms; force >= 0 takes
// position force mod (block size) of every block instead (a test hook: averaging the
// estimate over force = 0 .. m-1 gives every walker's e_x exactly when m divides the
// number of remaining walkers).  *nsel = |sel|; st gets the counts.
__global__ __launch_bounds__(1024) void k_cv_select(const int* __restrict__ live, const int* __restrict__ nlive,
                                                    const unsigned char* __restrict__ risky, int W, int m,
                                                    uint64_t seed, uint64_t draw, int force, int* __restrict__ tame,
                                                    int* __restrict__ sel, int* __restrict__ nsel,
                                                    float* __restrict__ pinv, double* __restrict__ st) {
  __shared__ int wr[16], wt[16];
  __shared__ int tot_r, tot_t;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwv = blockDim.x >> 6;
  for (int w = tid; w < W; w += blockDim.x) pinv[w] = 0.f;
  const int nl = *nlive;
  int off_r = 0, off_t = 0;
  for (int c0 = 0; c0 < nl; c0 += blockDim.x) {
    const int i = c0 + tid;
    const int w = i < nl ? live[i] : 0;
    const bool r = i < nl && risky && risky[w];
    const bool t = i < nl && !r;
    const unsigned long long mr = __ballot(r), mt = __ballot(t);
    const unsigned long long below = (1ull << lane) - 1ull;
    if (lane == 0) { wr[wave] = __popcll(mr); wt[wave] = __popcll(mt); }
    __syncthreads();
    int br = 0, bt = 0, sr = 0, stt = 0;
    for (int q = 0; q < nwv; ++q) {
      if (q < wave) { br += wr[q]; bt += wt[q]; }
      sr += wr[q];
      stt += wt[q];
    }
    if (r) sel[off_r + br + __popcll(mr & below)] = w;
    if (t) tame[off_t + bt + __popcll(mt & below)] = w;
    __syncthreads();
    off_r += sr;
    off_t += stt;
  }
  if (tid == 0) { tot_r = off_r; tot_t = off_t; }
  __syncthreads();   // pinv cleared, sel / tame complete
  const int nr = tot_r, nt = tot_t, nb = (nt + m - 1) / m;
  for (int i = tid; i < nr; i += blockDim.x) pinv[sel[i]] = 1.f;
  for (int b = tid; b < nb; b += blockDim.x) {
    const int b0 = b * m, bs = min(m, nt - b0);
    int pos;
    if (force >= 0) {
      pos = force % bs;
    } else {
      uint32_t c[4] = {(uint32_t)b, (uint32_t)draw, (uint32_t)(draw >> 32), 0x63760001u};
      philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
      const double u = (double)((((uint64_t)c[0] << 32) | c[1]) >> 11) * 0x1.0p-53;   // [0, 1)
      pos = min(bs - 1, (int)(u * bs));
    }
    const int k = tame[b0 + pos];
    sel[nr + b] = k;
    pinv[k] = (float)bs;
  }
  if (tid == 0) {
    *nsel = nr + nb;
    st[SS_NRISK] = nr;
    st[SS_NRAND] = nb;
    st[SS_NEXACT] = nr + nb;
  }
}
void launch_cv_select(const DevState& s, const unsigned char* risky, int m, uint64_t seed, uint64_t draw, int force,
                      int* tame, int* sel, int* nsel, float* pinv, hipStream_t st) {
  hipLaunchKernelGGL(k_cv_select, dim3(1), dim3(1024), 0, st, s.live, s.nlive, risky, s.W, m, seed, draw, force, tame,
                     sel, nsel, pinv, s.stats);
}

// Residual statistics of the random part of the exact set (sel[nrisk .. nsel)): RMS and
// mean of r = (S - soff) - (E_K - E_J), and the subset-sampling variance of the weighted
// mean energy, sum pinv (pinv - 1) (w d)^2 / (sum w)^2 (d = e_x - e_s of the clipped
// energies).  soff is the offset this measurement used.
__global__ __launch_bounds__(256) void k_cv_stats(const double* __restrict__ S, const double* __restrict__ EK,
                                                  const double* __restrict__ EJ, const double* __restrict__ D,
                                                  const float* __restrict__ pinv, const double* __restrict__ w,
                                                  const int* __restrict__ sel, const int* __restrict__ nsel, int W,
                                                  double* __restrict__ st) {
  __shared__ double red[16];
  const int nr = (int)st[SS_NRISK], ns = *nsel;
  const double soff = st[SS_CVOFF];
  double r2 = 0.0, rm = 0.0, wr2 = 0.0, ws = 0.0;
  for (int q = nr + (int)threadIdx.x; q < ns; q += blockDim.x) {
    const int k = sel[q];
    const double r = S[k] - soff - (EK[k] - EJ[k]);
    r2 += r * r;
    rm += r;
    const double p = pinv[k], wd = w[k] * D[k];
    wr2 += p * (p - 1.0) * wd * wd;
  }
  for (int q = threadIdx.x; q < W; q += blockDim.x) ws += w[q];
  r2 = block_sum(r2, red);
  rm = block_sum(rm, red);
  wr2 = block_sum(wr2, red);
  ws = block_sum(ws, red);
  if (threadIdx.x == 0) {
    const int nrand = ns - nr;
    st[SS_CVRMS] = nrand ? sqrt(r2 / nrand) : 0.0;
    st[SS_CVMEAN] = nrand ? rm / nrand : 0.0;
    st[SS_CVVAR] = ws > 0.0 ? wr2 / (ws * ws) : 0.0;
  }
}
// the running offset moves by rate x this measurement's mean residual; only the next
// measurement uses it, so every estimate stays unbiased
__global__ void k_cv_offset(double* st, double rate) {
  if (threadIdx.x == 0 && st[SS_NRAND] > 0.0) st[SS_CVOFF] += rate * st[SS_CVMEAN];
}
void launch_cv_stats(const DevState& s, const double* S, const double* EK, const double* EJ, const double* D,
                     const float* pinv, const int* sel, const int* nsel, hipStream_t st) {
  hipLaunchKernelGGL(k_cv_stats, dim3(1), dim3(256), 0, st, S, EK, EJ, D, pinv, s.weights, sel, nsel, s.W, s.stats);
}
void launch_cv_offset(const DevState& s, double rate, hipStream_t st) {
  hipLaunchKernelGGL(k_cv_offset, dim3(1), dim3(64), 0, st, s.stats, rate);
}

// ---------------------------------------------------------------- risk stratum
// The fraction risk of the live walkers whose Coulomb energy E_J lies farthest from the
// live walkers' median (ties: lower walker index first), as risky[w] = 1.  Two stable
// radix sorts of all W walkers (dead walkers keyed +inf, so they sort last): E_J gives
// the median (the (n/2)-th smallest of the n live values), then -|E_J - median| gives
// the stratum.
__global__ void k_risk_keys(const double* ej, const double* w, int W, const double* sorted, const int* nlive,
                            double* keys, int* idx, unsigned char* risky, int pass) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= W) return;
  const bool live = w[q] != 0.0;
  double k = INFINITY;
  if (live) {
    if (pass == 0) {
      k = ej[q];
    } else {
      const double med = sorted[*nlive / 2];
      k = -fabs(ej[q] - med);
    }
  }
  keys[q] = k;
  idx[q] = q;
  if (risky) risky[q] = 0;
}
__global__ void k_risk_mark(const int* idx_sorted, const int* nlive, double risk, unsigned char* risky) {
  const int nl = *nlive;
  const int nr = min(nl, (int)ceil(risk * nl));
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nr; i += gridDim.x * blockDim.x) risky[idx_sorted[i]] = 1;
}
size_t risk_sort_bytes(int W) {
  size_t bytes = 0;
  hcheck(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const double*)nullptr, (double*)nullptr,
                                                 (const int*)nullptr, (int*)nullptr, W), "radix sort size");
  return bytes;
}
void launch_risk_split(const DevState& s, const double* ej, double risk, RiskSort& rs, unsigned char* risky,
                       hipStream_t st) {
  const unsigned g = cdivu(s.W, 256);
  hipLaunchKernelGGL(k_risk_keys, dim3(g), dim3(256), 0, st, ej, s.weights, s.W, nullptr, s.nlive, rs.kin, rs.iin,
                     nullptr, 0);
  size_t bytes = rs.tmp_bytes;
  hcheck(hipcub::DeviceRadixSort::SortPairs(rs.tmp, bytes, rs.kin, rs.kout, rs.iin, rs.iout, s.W, 0, 64, st),
              "radix sort");
  hipLaunchKernelGGL(k_risk_keys, dim3(g), dim3(256), 0, st, ej, s.weights, s.W, rs.kout, s.nlive, rs.kin, rs.iin,
                     risky, 1);
  bytes = rs.tmp_bytes;
  hcheck(hipcub::DeviceRadixSort::SortPairs(rs.tmp, bytes, rs.kin, rs.kout, rs.iin, rs.iout, s.W, 0, 64, st),
              "radix sort");
  hipLaunchKernelGGL(k_risk_mark, dim3(g), dim3(256), 0, st, rs.iout, s.nlive, risk, risky);
}

}  // namespace afq
