// HIP kernels of the phaseless-AFQMC walker step for gfx950 (FP64 path).
//
// Every dense contraction is a real GEMM on the FP64 MFMA tile engine
// (afq_device.hpp) with loaders that read the operand in its storage layout:
//   VHS           P[(w,c), t]  = sum_g field[w][g][c] Lp[g][t]          (DQMC/DQMCWalker.cpp:406-421)
//   one-body      E psi, batched over walkers folded into columns        (DQMC/DQMCWalker.cpp:482-491)
//   Taylor term   V t with complex V embedded as [A_re | A_im] x [[B_re,B_im],[-B_im,B_re]]
//                                                                        (DQMC/DQMCWalker.cpp:424-431)
//   Green         S = Phi^T psi, S^-1 by Gauss-Jordan in LDS, theta = psi S^-1
//                                                                        (DQMC/RHF.cpp:27-61,104-131)
//   exchange      f = R_g theta per (g, walker) block, sum_ij f_ij f_ji reduced from
//                 the LDS-staged output tile without writing f           (DQMC/UHF.cpp:94-100)
#include <float.h>

#include <algorithm>
#include <utility>

#include "afq_device.hpp"
#include "afq_internal.hpp"
#include <type_traits>

namespace afq {

static inline unsigned cdivu(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

// live[0 .. *count) = the walkers of nonzero weight, ascending (one workgroup)
__device__ __forceinline__ void k_live_list_body(const uint3 bid_, const uint3 gdim_, const double* weights, int W, int* live, int* count) {
  __shared__ int wtot[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int offset = 0;
  for (int c0 = 0; c0 < W; c0 += 1024) {
    const int w = c0 + (int)threadIdx.x;
    const bool on = w < W && weights[w] != 0.0;
    const unsigned long long m = __ballot(on);
    const int pre = __popcll(m & ((1ull << lane) - 1ull));
    if (lane == 0) wtot[wave] = __popcll(m);
    __syncthreads();
    int base = 0, tot = 0;
    for (int q = 0; q < 16; ++q) {
      if (q < wave) base += wtot[q];
      tot += wtot[q];
    }
    if (on) live[offset + base + pre] = w;
    __syncthreads();
    offset += tot;
  }
  if (threadIdx.x == 0) *count = offset;
}
struct F_k_live_list {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_live_list_body(b, g, a...);
  }
};
__global__ __launch_bounds__(1024) void k_live_list(const double* weights, int W, int* live, int* count) {
  k_live_list_body(blockIdx3(), gridDim3(), weights, W, live, count);
}
void launch_live_list(const DevState& s, hipStream_t st) {
  afq::glaunch<F_k_live_list>(k_live_list, dim3(1), dim3(1024), 0, st, s.weights, s.W, s.live, s.nlive);
}

// ------------------------------------------------------------------ fields
// Philox4x32-10 (afq_device.hpp), counter = (pair index, step lo, step hi, walker),
// key = seed; two 53-bit uniforms per call, Box-Muller to two normals.
__device__ inline double philox_normal(uint64_t seed, int w, uint64_t step, int g) {
  uint32_t c[4] = {(uint32_t)(g >> 1), (uint32_t)step, (uint32_t)(step >> 32), (uint32_t)w};
  philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
  const uint64_t a = ((uint64_t)c[0] << 32) | c[1], b = ((uint64_t)c[2] << 32) | c[3];
  const double u1 = ((double)(a >> 11) + 1.0) * 0x1.0p-53;  // (0, 1]
  const double u2 = (double)(b >> 11) * 0x1.0p-53;          // [0, 1)
  const double r = sqrt(-2.0 * log(u1));
  double sn, cs;
  sincospi(2.0 * u2, &sn, &cs);
  return (g & 1) ? r * sn : r * cs;
}

// field loop of DQMC/DQMCWalker.cpp:451-457 for every live walker
__device__ __forceinline__ void k_fields_body(const uint3 bid_, const uint3 gdim_, const double* fb, const double* mf, const double* draws,
                                                const double* weights, double* fields, double* sft,
                                                int G, double dt, int ref_compat, uint64_t seed,
                                                uint64_t step, const unsigned long long* step_dev,
                                                unsigned long long* counters) {
  __shared__ double red[16];
  const int w = bid_.x;
  // the step's counters, which its weight update adds to
  if (w == 0 && threadIdx.x < 2) counters[threadIdx.x] = 0ull;
  if (weights[w] <= 1e-8) return;
  if (step_dev) step = *step_dev;  // replayed graphs read the step counter from memory
  const double sq = sqrt(dt);
  double sh_re = 0, sh_im = 0, ft_re = 0, ft_im = 0;
  for (int g = threadIdx.x; g < G; g += blockDim.x) {
    const double x = draws ? draws[(int64_t)w * G + g] : philox_normal(seed, w, step, g);
    const double fr = fb[(int64_t)w * 2 * G + 2 * g], fi = fb[(int64_t)w * 2 * G + 2 * g + 1];
    const double mr = mf[2 * g], mi = mf[2 * g + 1];
    // s = -sqrt(dt) (i fb - mf)
    const double s_re = -sq * (-fi - mr), s_im = -sq * (fr - mi);
    double p_re = x - s_re, p_im = -s_im;
    // shift += (x - s) mf ; fbTerm += x s - s^2/2
    sh_re += p_re * mr - p_im * mi;
    sh_im += p_re * mi + p_im * mr;
    ft_re += x * s_re - 0.5 * (s_re * s_re - s_im * s_im);
    ft_im += x * s_im - s_re * s_im;
    if (ref_compat) { p_re = (double)(float)p_re; p_im = (double)(float)p_im; }
    fields[(int64_t)w * 2 * G + 2 * g] = p_re;
    fields[(int64_t)w * 2 * G + 2 * g + 1] = p_im;
  }
  sh_re = block_sum(sh_re, red);
  sh_im = block_sum(sh_im, red);
  ft_re = block_sum(ft_re, red);
  ft_im = block_sum(ft_im, red);
  if (threadIdx.x == 0) {
    sft[4 * w] = sh_re; sft[4 * w + 1] = sh_im; sft[4 * w + 2] = ft_re; sft[4 * w + 3] = ft_im;
  }
}
struct F_k_fields {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_fields_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_fields(const double* fb, const double* mf, const double* draws,
                                                const double* weights, double* fields, double* sft,
                                                int G, double dt, int ref_compat, uint64_t seed,
                                                uint64_t step, const unsigned long long* step_dev,
                                                unsigned long long* counters) {
  k_fields_body(blockIdx3(), gridDim3(), fb, mf, draws, weights, fields, sft, G, dt, ref_compat, seed, step, step_dev, counters);
}

void launch_fields(const DevState& s, const double* draws, uint64_t seed, uint64_t step, hipStream_t st) {
  afq::glaunch<F_k_fields>(k_fields, dim3(s.W), dim3(256), 0, st, s.fb, s.mf, draws, s.weights, s.fields,
                     s.sft, s.G, s.dt, (int)s.ref_compat, seed, step, s.d_step, s.ncap);
}

// ------------------------------------------------------------------ propagation
// out = E * src for determinant d of every walker (walkers folded into columns).
struct ExpA {
  const double* E; int N; int row0;
  __device__ double operator()(int r, int k) const {
    const int i = row0 + r;
    return (i < N && k < N) ? E[(int64_t)i * N + k] : 0.0;
  }
};
struct DetColsB {  // B(k, q) = src[w][det d][k][cc], q = w*2n + cc
  const double* src; int64_t wstride, doff; int N, n2, q0, ncol;
  __device__ double operator()(int k, int c) const {
    const int q = q0 + c;
    if (q >= ncol || k >= N) return 0.0;
    const int w = q / n2, cc = q - w * n2;
    return src[(int64_t)w * wstride + doff + (int64_t)k * n2 + cc];
  }
};
constexpr int EX_BM = 64, EX_BN = 128;
// mode 0: dst1 = dst2 = E src (start of the Taylor series); mode 1: dst1 = E src for live walkers
__device__ __forceinline__ void k_expmul_body(const uint3 bid_, const uint3 gdim_, const double* E, const double* src, double* dst1,
                                                double* dst2, const double* weights, int N, int n,
                                                int W, int64_t wstride, int64_t doff, int mode, int gridx,
                                                int gridy) {
  using Eng = MmaF64<EX_BM, EX_BN, 2, 2, false, true>;
  __shared__ double lds[Eng::LDS_DOUBLES];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, 1, gridy);
  const int row0 = tl.y * EX_BM, q0 = tl.x * EX_BN;
  const int n2 = 2 * n, ncol = W * n2;
  Eng e;
  e.run(ExpA{E, N, row0}, DetColsB{src, wstride, doff, N, n2, q0, ncol}, N, lds);
  e.store([&](int r, int c, double v) {
    const int i = row0 + r, q = q0 + c;
    if (i >= N || q >= ncol) return;
    const int w = q / n2, cc = q - w * n2;
    if (weights[w] <= 1e-8) return;
    const int64_t a = (int64_t)w * wstride + doff + (int64_t)i * n2 + cc;
    dst1[a] = v;
    if (mode == 0) dst2[a] = v;
  });
}
struct F_k_expmul {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_expmul_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_expmul(const double* E, const double* src, double* dst1,
                                                double* dst2, const double* weights, int N, int n,
                                                int W, int64_t wstride, int64_t doff, int mode, int gridx,
                                                int gridy) {
  k_expmul_body(blockIdx3(), gridDim3(), E, src, dst1, dst2, weights, N, n, W, wstride, doff, mode, gridx, gridy);
}

// t_dst = (V t_src)/p, acc += t_dst for one walker per blockIdx.z; V = i sqrt(dt) (P_re + i P_im)
struct VA {  // [A_re | A_im], A_re = -sq P_im, A_im = sq P_re (full N x N rows)
  const double* Pre; const double* Pim; int N; int row0; double sq;
  __device__ double operator()(int r, int k) const {
    const int i = row0 + r;
    if (i >= N || k >= 2 * N) return 0.0;
    return k < N ? -sq * Pim[(int64_t)i * N + k] : sq * Pre[(int64_t)i * N + (k - N)];
  }
};
struct TB {  // [[B_re, B_im], [-B_im, B_re]] over the walker's propagated dets, interleaved cols
  const double* src; int N; int n2a, n2b; int64_t offb; int q0, ncol;
  __device__ double operator()(int k, int c) const {
    const int q = q0 + c;
    if (q >= ncol || k >= 2 * N) return 0.0;
    const double* base;
    int n2, cl;
    if (q < n2a) { base = src; n2 = n2a; cl = q; }
    else { base = src + offb; n2 = n2b; cl = q - n2a; }
    if (k < N) return base[(int64_t)k * n2 + cl];
    const int comp = cl & 1, j2 = cl - comp;
    const double* row = base + (int64_t)(k - N) * n2 + j2;
    return comp ? row[0] : -row[1];
  }
};
// One walker's V t for a BM x BN tile of (orbital row, determinant column) through
// the generic engine; used when a walker has at most 64 electrons (k_taylor below
// serves the wider determinants).
template <int VM_BM, int VM_BN, int WVM, int WVN>
__device__ __forceinline__ void k_vmul_body(const uint3 bid_, const uint3 gdim_, const double* P, const double* tsrc, double* tdst,
                                              double* acc, const double* weights, int N, int64_t T,
                                              int n2a, int n2b, int64_t offb, int64_t wstride,
                                              double sq, double inv_p, int gridx, int gridy, int W) {
  using Eng = MmaF64<VM_BM, VM_BN, WVM, WVN, false, true>;
  __shared__ double lds[Eng::LDS_DOUBLES];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, W, gridy);
  const int w = tl.z;
  if (weights[w] <= 1e-8) return;
  const int row0 = tl.y * VM_BM, q0 = tl.x * VM_BN;
  const int ncol = n2a + n2b;
  const double* Pre = P + (int64_t)(2 * w) * N * N;
  const double* Pim = Pre + (int64_t)N * N;
  const double* src = tsrc + (int64_t)w * wstride;
  Eng e;
  e.run(VA{Pre, Pim, N, row0, sq}, TB{src, N, n2a, n2b, offb, q0, ncol}, 2 * N, lds);
  double* dst = tdst + (int64_t)w * wstride;
  double* ac = acc + (int64_t)w * wstride;
  e.store([&](int r, int c, double v) {
    const int i = row0 + r, q = q0 + c;
    if (i >= N || q >= ncol) return;
    const int64_t a = q < n2a ? (int64_t)i * n2a + q : offb + (int64_t)i * n2b + (q - n2a);
    const double x = v * inv_p;
    dst[a] = x;
    ac[a] += x;
  });
}
template <int VM_BM, int VM_BN, int WVM, int WVN>
struct F_k_vmul {
  static constexpr int NT = 64 * WVM * WVN, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_vmul_body<VM_BM, VM_BN, WVM, WVN>(b, g, a...);
  }
};
template <int VM_BM, int VM_BN, int WVM, int WVN>
__global__ __launch_bounds__(64 * WVM * WVN) void k_vmul(const double* P, const double* tsrc, double* tdst,
                                              double* acc, const double* weights, int N, int64_t T,
                                              int n2a, int n2b, int64_t offb, int64_t wstride,
                                              double sq, double inv_p, int gridx, int gridy, int W) {
  k_vmul_body<VM_BM, VM_BN, WVM, WVN>(blockIdx3(), gridDim3(), P, tsrc, tdst, acc, weights, N, T, n2a, n2b, offb, wstride, sq, inv_p, gridx, gridy, W);
}

// One Taylor product t_dst = (i sq P) t_src / p (acc += t_dst) for a 128-row x
// 128-complex-column tile of one walker, 8 waves (2 x 4) on FP64 MFMA.  The complex
// product is the real GEMM [A_re | A_im] [[T_re, T_im], [-T_im, T_re]] with
// A = i P (A_re = -P_im, A_im = P_re); each K slice covers 8 orbitals, i.e. 16
// real K rows: the P rows arrive as 16-byte pairs along k, the t rows as complex
// numbers, and the embedding (swap and sign) is applied while staging into LDS.
// The next slice is prefetched into registers while the current one multiplies.
constexpr int TY_BM = 128, TY_BNC = 128, TY_BN = 2 * TY_BNC, TY_KC = 8, TY_K = 2 * TY_KC;
constexpr int TY_LDA = TY_BM + 2, TY_LDB = TY_BN + 2;
template <bool PAIRS>
__device__ __forceinline__ void k_taylor_body(const uint3 bid_, const uint3 gdim_, const double* P, const double* tsrc, double* tdst, double* acc,
                                                const double* weights, int N, int na, int nb, int64_t offb,
                                                int64_t wstride, double scale, int gridx, int gridy, int W) {
  __shared__ double As[TY_K * TY_LDA];
  __shared__ double Bs[TY_K * TY_LDB];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, W, gridy);
  const int w = tl.z;
  if (weights[w] <= 1e-8) return;
  const int row0 = tl.y * TY_BM, q0 = tl.x * TY_BNC, ncolc = na + nb;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 2, wn = wave & 3;
  const double* Pre = P + (int64_t)(2 * w) * N * N;
  const double* Pim = Pre + (int64_t)N * N;
  const double* src = tsrc + (int64_t)w * wstride;
  // A: thread -> (row r = tid / 4, orbital pair kp = 2 (tid % 4)) of the slice
  const int ar = tid >> 2, akp = (tid & 3) * 2, ai = row0 + ar;
  // B: thread -> (orbital kk, complex column qc) for two elements e = tid, tid + 512
  double2 pa_re, pa_im, tb[2];
  auto fetch = [&](int k0) {
    const int k = k0 + akp;
    pa_re = double2{0.0, 0.0};
    pa_im = double2{0.0, 0.0};
    if (ai < N) {
      const int64_t o = (int64_t)ai * N + k;
      if (PAIRS && k + 1 < N) {
        pa_re = *reinterpret_cast<const double2*>(Pre + o);
        pa_im = *reinterpret_cast<const double2*>(Pim + o);
      } else {
        if (k < N) { pa_re.x = Pre[o]; pa_im.x = Pim[o]; }
        if (k + 1 < N) { pa_re.y = Pre[o + 1]; pa_im.y = Pim[o + 1]; }
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int e = tid + 512 * h, kk = e / TY_BNC, qc = e % TY_BNC;
      const int kr = k0 + kk, q = q0 + qc;
      tb[h] = double2{0.0, 0.0};
      if (kr < N && q < ncolc) {
        const double* rowp = q < na ? src + 2 * ((int64_t)kr * na + q) : src + 2 * (offb + (int64_t)kr * nb + (q - na));
        tb[h] = *reinterpret_cast<const double2*>(rowp);
      }
    }
  };
  auto stage = [&]() {
    // A_re = -P_im (rows 0..7 of the slice), A_im = P_re (rows 8..15)
    As[(akp + 0) * TY_LDA + ar] = -pa_im.x;
    As[(akp + 1) * TY_LDA + ar] = -pa_im.y;
    As[(TY_KC + akp + 0) * TY_LDA + ar] = pa_re.x;
    As[(TY_KC + akp + 1) * TY_LDA + ar] = pa_re.y;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int e = tid + 512 * h, kk = e / TY_BNC, qc = e % TY_BNC;
      Bs[kk * TY_LDB + 2 * qc] = tb[h].x;
      Bs[kk * TY_LDB + 2 * qc + 1] = tb[h].y;
      Bs[(TY_KC + kk) * TY_LDB + 2 * qc] = -tb[h].y;
      Bs[(TY_KC + kk) * TY_LDB + 2 * qc + 1] = tb[h].x;
    }
  };
  f64x4 c[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) c[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
  const int nst = (N + TY_KC - 1) / TY_KC;
  fetch(0);
  for (int st = 0; st < nst; ++st) {
    stage();
    __syncthreads();
    if (st + 1 < nst) fetch((st + 1) * TY_KC);
#pragma unroll
    for (int k4 = 0; k4 < TY_K / 4; ++k4) {
      const int kr = k4 * 4 + (lane >> 4);
      double a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kr * TY_LDA + wm * 64 + i * 16 + (lane & 15)];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[kr * TY_LDB + wn * 64 + j * 16 + (lane & 15)];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) c[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], c[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  double* dst = tdst + (int64_t)w * wstride;
  double* ac = acc + (int64_t)w * wstride;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = row0 + wm * 64 + i * 16 + (lane >> 4) + 4 * r;
        const int cr = wn * 64 + j * 16 + (lane & 15);  // real column in the tile
        const int q = q0 + (cr >> 1), comp = cr & 1;
        if (row < N && q < ncolc) {
          const int64_t a = (q < na ? 2 * ((int64_t)row * na + q) : 2 * (offb + (int64_t)row * nb + (q - na))) + comp;
          const double x = c[i][j][r] * scale;
          dst[a] = x;
          ac[a] += x;
        }
      }
}
template <bool PAIRS>
struct F_k_taylor {
  static constexpr int NT = 512, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_taylor_body<PAIRS>(b, g, a...);
  }
};
template <bool PAIRS>
__global__ __launch_bounds__(512) void k_taylor(const double* P, const double* tsrc, double* tdst, double* acc,
                                                const double* weights, int N, int na, int nb, int64_t offb,
                                                int64_t wstride, double scale, int gridx, int gridy, int W) {
  k_taylor_body<PAIRS>(blockIdx3(), gridDim3(), P, tsrc, tdst, acc, weights, N, na, nb, offb, wstride, scale, gridx, gridy, W);
}

// Split-BF16 Taylor series by Horner's rule: u <- t0 + (V u) sqrt(dt)/p for p = 5..1,
// starting from u = t0 = E psi, so that the last step leaves sum_{k<=5} V^k/k! t0.
// V = i sqrt(dt) P enters as the real matrix [A_re | A_im] = [-P_im | P_re] against
// [[u_re, u_im], [-u_im, u_re]], three MFMA passes hi*hi + hi*lo + lo*hi (x = hi + lo)
// with FP32 accumulation.  All operands arrive already split (VHS epilogue, k_expmul,
// previous Horner step) in orbital chunks of 16, so a K stage is one chunk: 16 orbitals
// = 32 real K = one v_mfma_f32_16x16x32_bf16, and its A and B slices are contiguous.
// Intermediate u are stored split; the last step adds the FP64 t0 and writes FP64.
// Tile: 32*MI orbital rows x 32*NI complex columns, 8 waves as 2 (rows) x 4 (columns).
// Tile: 32*MI orbital rows x 32*NI complex columns, 8 waves as 2 (rows) x 4 (columns);
// a stage holds CPS chunks (its loads prefetched into registers one stage ahead).
constexpr int TH_LDK = 40;
template <int MI, int NI, int CPS>
__device__ __forceinline__ void k_taylor_h_body(const uint3 bid_, const uint3 gdim_, const u16* Vh, const u16* Vl, const u16* Ui, u16* Uo,
                                                  const u16* T0b, const double* t0, double* out,
                                                  const double* weights, int N, int Nq, int na, int nb,
                                                  int64_t offb, int64_t wstride, float scale, int last,
                                                  int gridx, int gridy, int W) {
  constexpr int BM = 32 * MI, BN = 64 * NI, BNC = BN / 2, LDK = 32 * CPS + 8;
  constexpr int AV = 2 * BM * 4, AVT = (AV + 511) / 512;     // 16-B vectors per chunk: A
  constexpr int BV = 4 * BNC * 2, BVT = (BV + 511) / 512;    //                         B
  __shared__ __attribute__((aligned(16))) u16 As[2][BM * LDK];
  __shared__ __attribute__((aligned(16))) u16 Bs[2][BN * LDK];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, W, gridy);
  const int w = tl.z;
  if (weights[w] <= 1e-8) return;
  const int row0 = tl.y * BM, q0 = tl.x * BNC, ncolc = na + nb;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 2, wn = wave & 3;
  const int nch = Nq >> 4;
  const int64_t vper = (int64_t)nch * N * 32;     // one walker's V plane
  const int64_t uplane = (int64_t)ncolc * Nq;     // one u plane
  const u16* vh = Vh + (int64_t)w * vper;
  const u16* vl = Vl + (int64_t)w * vper;
  const u16* ui = Ui + (int64_t)w * 4 * uplane;
  uint4 ra[CPS][AVT], rb[CPS][BVT];
  auto fetch = [&](int ch0) {
#pragma unroll
    for (int cc = 0; cc < CPS; ++cc) {
      const int ch = ch0 + cc;
#pragma unroll
      for (int h = 0; h < AVT; ++h) {
        const int e = tid + 512 * h;
        ra[cc][h] = uint4{0u, 0u, 0u, 0u};
        if (e < AV && ch < nch) {
          const int pl = e / (BM * 4), r = (e >> 2) - pl * BM, v = e & 3, i = row0 + r;
          if (i < N) ra[cc][h] = *reinterpret_cast<const uint4*>((pl ? vl : vh) + ((int64_t)ch * N + i) * 32 + 8 * v);
        }
      }
#pragma unroll
      for (int h = 0; h < BVT; ++h) {
        const int e = tid + 512 * h;
        rb[cc][h] = uint4{0u, 0u, 0u, 0u};
        if (e < BV && ch < nch) {
          const int pl = e / (BNC * 2), rem = e - pl * (BNC * 2), q = q0 + (rem >> 1);
          if (q < ncolc)
            rb[cc][h] =
                *reinterpret_cast<const uint4*>(ui + pl * uplane + ((int64_t)ch * ncolc + q) * 16 + 8 * (rem & 1));
        }
      }
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int cc = 0; cc < CPS; ++cc) {
#pragma unroll
      for (int h = 0; h < AVT; ++h) {
        const int e = tid + 512 * h;
        if (e < AV) {
          const int pl = e / (BM * 4), r = (e >> 2) - pl * BM, v = e & 3;
          *reinterpret_cast<uint4*>(As[pl] + r * LDK + 32 * cc + 8 * v) = ra[cc][h];
        }
      }
#pragma unroll
      for (int h = 0; h < BVT; ++h) {
        const int e = tid + 512 * h;
        if (e < BV) {
          // plane pl = 2*comp + (lo); columns (q, re) = [u_re | -u_im], (q, im) = [u_im | u_re]
          const int pl = e / (BNC * 2), rem = e - pl * (BNC * 2), qc = rem >> 1, half = rem & 1;
          u16* dst = Bs[pl & 1] + 32 * cc;
          const uint4 x = rb[cc][h];
          if (pl < 2) {
            *reinterpret_cast<uint4*>(dst + (2 * qc) * LDK + 8 * half) = x;
            *reinterpret_cast<uint4*>(dst + (2 * qc + 1) * LDK + 16 + 8 * half) = x;
          } else {
            const uint4 nx = uint4{x.x ^ 0x80008000u, x.y ^ 0x80008000u, x.z ^ 0x80008000u, x.w ^ 0x80008000u};
            *reinterpret_cast<uint4*>(dst + (2 * qc + 1) * LDK + 8 * half) = x;
            *reinterpret_cast<uint4*>(dst + (2 * qc) * LDK + 16 + 8 * half) = nx;
          }
        }
      }
    }
  };
  f32x4 c[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) c[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nst = (nch + CPS - 1) / CPS;
  fetch(0);
  for (int st = 0; st < nst; ++st) {
    stage();
    __syncthreads();
    if (st + 1 < nst) fetch((st + 1) * CPS);
#pragma unroll
    for (int cc = 0; cc < CPS; ++cc) {
      const int koff = 32 * cc + 8 * (lane >> 4);
      bf16x8 b[2][NI];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          b[h][j] = *reinterpret_cast<const bf16x8*>(Bs[h] + (wn * 16 * NI + j * 16 + (lane & 15)) * LDK + koff);
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(As[0] + (wm * 16 * MI + i * 16 + (lane & 15)) * LDK + koff);
        const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(As[1] + (wm * 16 * MI + i * 16 + (lane & 15)) * LDK + koff);
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b[0][j], c[i][j], 0, 0, 0);
          c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b[1][j], c[i][j], 0, 0, 0);
          c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b[0][j], c[i][j], 0, 0, 0);
        }
      }
    }
    __syncthreads();
  }
  // lane holds rows 4*(lane/16) + r (r = 0..3) of column lane % 16: four consecutive
  // orbitals of one chunk
  const u16* t0w = T0b + (int64_t)w * 4 * uplane;
  u16* uo = Uo + (int64_t)w * 4 * uplane;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int rowb = row0 + wm * 16 * MI + i * 16 + 4 * (lane >> 4);
      const int cr = wn * 16 * NI + j * 16 + (lane & 15);
      const int q = q0 + (cr >> 1), comp = cr & 1;
      if (rowb >= N || q >= ncolc) continue;
      if (!last) {
        const int64_t o = 2 * comp * uplane + ((int64_t)(rowb >> 4) * ncolc + q) * 16 + (rowb & 15);
        const uint2 th = *reinterpret_cast<const uint2*>(t0w + o);
        const uint2 tlo = *reinterpret_cast<const uint2*>(t0w + o + uplane);
        const unsigned hw[4] = {th.x & 0xffffu, th.x >> 16, th.y & 0xffffu, th.y >> 16};
        const unsigned lw[4] = {tlo.x & 0xffffu, tlo.x >> 16, tlo.y & 0xffffu, tlo.y >> 16};
        float x[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          x[r] = bf_bits2f((u16)hw[r]) + bf_bits2f((u16)lw[r]) + c[i][j][r] * scale;
          if (rowb + r >= N) x[r] = 0.f;   // orbital pads stay zero
        }
        uint2 oh, ol;
        split4_bf16(x, oh, ol);
        *reinterpret_cast<uint2*>(uo + o) = oh;
        *reinterpret_cast<uint2*>(uo + o + uplane) = ol;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = rowb + r;
          if (row >= N) break;
          const int64_t a = (q < na ? 2 * ((int64_t)row * na + q) : 2 * (offb + (int64_t)row * nb + (q - na))) + comp;
          out[(int64_t)w * wstride + a] = t0[(int64_t)w * wstride + a] + (double)c[i][j][r] * (double)scale;
        }
      }
    }
}
template <int MI, int NI, int CPS>
struct F_k_taylor_h {
  static constexpr int NT = 512, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_taylor_h_body<MI, NI, CPS>(b, g, a...);
  }
};
template <int MI, int NI, int CPS>
__global__ __launch_bounds__(512) void k_taylor_h(const u16* Vh, const u16* Vl, const u16* Ui, u16* Uo,
                                                  const u16* T0b, const double* t0, double* out,
                                                  const double* weights, int N, int Nq, int na, int nb,
                                                  int64_t offb, int64_t wstride, float scale, int last,
                                                  int gridx, int gridy, int W) {
  k_taylor_h_body<MI, NI, CPS>(blockIdx3(), gridDim3(), Vh, Vl, Ui, Uo, T0b, t0, out, weights, N, Nq, na, nb, offb, wstride, scale, last, gridx, gridy, W);
}

// The whole split-BF16 propagation of one walker's block of columns in one workgroup:
//   x <- E (sum_{k<=5} V^k / k!) E x,   E = I + D,
// (DQMC/DQMCWalker.cpp:424-431,482-491) with the Taylor sum by Horner's rule.  The block
// (QB = 8*CT complex columns of the na + nb propagated ones, all N orbitals) stays in LDS
// for the whole propagation, split (hi, lo) in the compact layout
//   u[hl][re/im][chunk][q][16 orbitals]
// and is the B operand of every product; the A operands (D = E - I, and V = the split
// [-P_im | P_re] chunks of the VHS) are read straight from global memory into MFMA
// fragments, since each wave owns its own rows (wave v: row tiles v, v+8, .., all CT
// column tiles) and no other wave of the workgroup reads them.  So a product needs no
// barrier; one step of the series costs two.  Eight waves, two per SIMD: the A fragments
// run one or two K stages ahead in two or three register sets, and a product's first
// stages are requested before the barrier that precedes it.  The first
// factor t0 = E x is kept in FP32 registers at each lane's output positions; Horner's
// steps u <- t0 + (V u) sqrt(dt)/p go back to LDS split, and the result leaves as FP64
// after the last E.  The blocks of one walker run back to back on one XCD, so V and D
// stream from HBM about once per product for all of them.  Walkers at or below the
// propagation threshold are skipped.
constexpr int PS_WAVES = 8;
constexpr int PS_MT_MAX = 3;   // row tiles per wave: N <= 16 * PS_WAVES * PS_MT_MAX = 384
template <int MT, int CT>
struct PropShape {
  static constexpr int QB = 8 * CT;                     // complex columns per block
  // orbital chunks of 16 held in LDS: the N orbitals (at most PS_WAVES MT chunks) and
  // zero chunks for the stages a product's loop adds past its end
  static constexpr int NCH = PS_WAVES * MT + 4;
  static constexpr int PLANE = NCH * QB * 16 + 8;       // u16 per plane (+ 16 B against bank aliasing)
  static constexpr int LDS_U16 = 4 * PLANE;
};
template <int MT, int CT>
__device__ __forceinline__ void k_prop_split_body(const uint3 bid_, const uint3 gdim_, const u16* __restrict__ Vh, const u16* __restrict__ Vl,
                                                                 const u16* __restrict__ Dh, const u16* __restrict__ Dl,
                                                                 const double* src, double* dst, const double* weights,
                                                                 int N, int Nd, int na, int nb, int64_t offb,
                                                                 int64_t wstride, float sq, int nblk, int W) {
  using S = PropShape<MT, CT>;
  constexpr int QB = S::QB, PLANE = S::PLANE, NT = 64 * PS_WAVES;
  __shared__ __attribute__((aligned(16))) u16 u[S::LDS_U16];   // [hi re, hi im, lo re, lo im]
  const TileId tl = tile_id_at(bid_.x, nblk, 1, W, 1);
  const int w = tl.z, blk = tl.x;
  if (weights[w] <= 1e-8) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int RT = (N + 15) >> 4;            // row tiles of 16 orbitals
  const int nch = RT;                      // V chunks (16 orbitals each)
  const int nks = (N + 31) >> 5;           // D steps (32 orbitals each)
  const int ncolc = na + nb, q0 = blk * QB;
  const int64_t vper = (int64_t)nch * N * 32;
  const u16* vh = Vh + (int64_t)w * vper;
  const u16* vl = Vl + (int64_t)w * vper;
  const double* xs = src + (int64_t)w * wstride;
  double* xd = dst + (int64_t)w * wstride;

  for (int e = tid; e < S::LDS_U16 / 8; e += NT) reinterpret_cast<uint4*>(u)[e] = uint4{0u, 0u, 0u, 0u};

  // this lane's output positions: rows 16 rt + 4 (lane >> 4) + r of column 16 j + (lane & 15)
  const int cl = lane & 15, kh = lane >> 4;
  int rt[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) rt[m] = wave + PS_WAVES * m;
  // FP64 offset of (row, this lane's column of column tile j) in the walker: cb[j] + row rs[j]
  int cb[CT], rs[CT];
  auto col_setup = [&](int qb) {
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int q = qb + 8 * j + (cl >> 1), comp = cl & 1;
      cb[j] = q < na ? 2 * q + comp : (int)(2 * (offb + q - na)) + comp;
      rs[j] = q < ncolc ? (q < na ? 2 * na : 2 * nb) : -1;   // -1: padding column
    }
  };
  col_setup(q0);
  auto valid = [&](int row, int j) { return row < N && rs[j] >= 0; };
  // LDS offset (u16) of 4 consecutive orbitals row.. of column q in plane (hl, comp)
  auto uoff = [&](int hl, int comp, int row, int q) { return (2 * hl + comp) * PLANE + ((row >> 4) * QB + q) * 16 + (row & 15); };

  float T[MT][CT][4];
  f32x4 acc[MT][CT];
  __syncthreads();
  // x: FP32 copy at the output positions, split into LDS
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int rb = 16 * rt[m] + 4 * kh;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        T[m][j][r] = (rt[m] < RT && valid(rb + r, j)) ? (float)xs[cb[j] + (int64_t)(rb + r) * rs[j]] : 0.f;
    }
  auto put = [&]() {   // T (or its Horner update in T) -> u, split
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (rt[m] >= RT) continue;   // wave-uniform
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        const int c = 16 * j + cl, rb = 16 * rt[m] + 4 * kh;
        float t[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) t[r] = rb + r < N ? T[m][j][r] : 0.f;   // orbital pads of u stay zero
        uint2 oh, ol;
        split4_bf16(t, oh, ol);
        *reinterpret_cast<uint2*>(u + uoff(0, c & 1, rb, c >> 1)) = oh;
        *reinterpret_cast<uint2*>(u + uoff(1, c & 1, rb, c >> 1)) = ol;
      }
    }
  };
  auto zero_acc = [&]() {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto mma3 = [&](const bf16x8* ah, const bf16x8* al, const bf16x8* bh, const bf16x8* bl) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (rt[m] >= RT) continue;   // wave-uniform
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[m], bh[j], acc[m][j], 0, 0, 0);
        acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[m], bl[j], acc[m][j], 0, 0, 0);
        acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[m], bh[j], acc[m][j], 0, 0, 0);
      }
    }
  };
  // A fragments straight from global memory into one of
  // NS register sets, stage k in set k % NS: three sets (loads two stages ahead) where
  // the registers allow, else two
  // (a wave-uniform row-tile base plus one 32-bit per-lane offset per operand, so that the
  // loads take a scalar base and the offsets cost one VGPR each)
  constexpr int NS = MT * CT >= 9 ? 2 : 3;
  bf16x8 Ah[NS][MT], Al[NS][MT];
  // The loads are unconditional (no branch, so the compiler can count them when it waits
  // for a stage): rows past N, and the row tiles a wave does not have, read row N - 1
  // instead, and the MFMA rows they feed never reach LDS or the output.
  unsigned doff[MT], voff[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = min(16 * rt[m] + cl, N - 1);
    doff[m] = (unsigned)(row * Nd + 8 * kh);
    voff[m] = (unsigned)(row * 32 + 8 * kh);
  }
  auto loadA = [&](const u16* hp, const u16* lp, const unsigned* off, int64_t koffs, bf16x8* h, bf16x8* l) {
    const u16* hb = hp + koffs;   // wave-uniform
    const u16* lb = lp + koffs;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      h[m] = *reinterpret_cast<const bf16x8*>(hb + off[m]);
      l[m] = *reinterpret_cast<const bf16x8*>(lb + off[m]);
    }
  };
  // D product: 32-orbital stages, A rows from Dh/Dl (pitch Nd), B = u without sign flips
  auto loadD = [&](int ks, int set) { loadA(Dh, Dl, doff, 32 * (int64_t)ks, Ah[set], Al[set]); };
  auto dstep = [&](int ks, int set) {
    const int k = 32 * ks + 8 * kh;
    bf16x8 bh[CT], bl[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int c = 16 * j + cl;
      bh[j] = *reinterpret_cast<const bf16x8*>(u + uoff(0, c & 1, k, c >> 1));
      bl[j] = *reinterpret_cast<const bf16x8*>(u + uoff(1, c & 1, k, c >> 1));
    }
    mma3(Ah[set], Al[set], bh, bl);
  };
  // V product: a chunk's 32 K are [16 orbitals of -P_im | 16 of P_re], against B column
  // (q, re) = [u_re | -u_im] and (q, im) = [u_im | u_re]
  const int sgn = kh >> 1, koff = 8 * (kh & 1);
  const unsigned nmask = ((cl & 1) == 0 && sgn) ? 0x80008000u : 0u;   // lanes holding -u_im
  auto loadV = [&](int ch, int set) { loadA(vh, vl, voff, (int64_t)ch * N * 32, Ah[set], Al[set]); };
  auto vstep = [&](int ch, int set) {
    bf16x8 bh[CT], bl[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int c = 16 * j + cl, comp = c & 1;
      const int o = uoff(0, comp ^ sgn, 16 * ch + koff, c >> 1);
      uint4 xh = *reinterpret_cast<const uint4*>(u + o);
      uint4 xl = *reinterpret_cast<const uint4*>(u + o + 2 * PLANE);
      xh = uint4{xh.x ^ nmask, xh.y ^ nmask, xh.z ^ nmask, xh.w ^ nmask};
      xl = uint4{xl.x ^ nmask, xl.y ^ nmask, xl.z ^ nmask, xl.w ^ nmask};
      bh[j] = *reinterpret_cast<const bf16x8*>(&xh);
      bl[j] = *reinterpret_cast<const bf16x8*>(&xl);
    }
    mma3(Ah[set], Al[set], bh, bl);
  };
  // one product over n stages whose stages 0 .. NS-2 are already requested (sets 0 ..
  // NS-2).  The loop is unrolled by NS (every set index a constant) and has no branch at
  // all, so the compiler can count the loads in flight when it waits for a stage: n is
  // rounded up to a multiple of NS, and the stages past n re-read the last A stage
  // against the zero orbital pads of u (NCH leaves room for them), adding nothing.
  auto product = [&](int n, auto load, auto step) {
    zero_acc();
    const int np = (n + NS - 1) / NS * NS;
    for (int k = 0; k < np; k += NS) {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        load(min(k + i + NS - 1, n - 1), (i + NS - 1) % NS);
        step(k + i, i);
      }
    }
  };
  auto preD = [&]() {
#pragma unroll
    for (int i = 0; i + 1 < NS; ++i) loadD(min(i, nks - 1), i);
  };
  auto preV = [&]() {
#pragma unroll
    for (int i = 0; i + 1 < NS; ++i) loadV(min(i, nch - 1), i);
  };

  put();
  preD();
  __syncthreads();
  product(nks, loadD, dstep);    // t0 = x + D x
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) T[m][j][r] += acc[m][j][r];
  preV();
  __syncthreads();
  put();
  __syncthreads();
  for (int p = 5; p >= 1; --p) {
    product(nch, loadV, vstep);
    if (p > 1) preV();
    else preD();
    __syncthreads();
    const float f = sq / (float)p;
    if (p > 1) {
      // u <- t0 + (V u) f: T keeps t0, the update goes to LDS through T's slot
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float t0 = T[m][j][r];
            T[m][j][r] = t0 + acc[m][j][r] * f;
            acc[m][j][r] = t0;
          }
      put();
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) T[m][j][r] = acc[m][j][r];
    } else {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) T[m][j][r] += acc[m][j][r] * f;
      put();
    }
    __syncthreads();
  }
  product(nks, loadD, dstep);    // E y = y + D y
  // the column offsets again from scratch (opaque to the compiler), so that the
  // prologue's addresses are not kept live through the whole kernel
  int q0o = q0;
  asm volatile("" : "+v"(q0o));
  col_setup(q0o);
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (rt[m] >= RT) continue;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int rb = 16 * rt[m] + 4 * kh;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (valid(rb + r, j)) xd[cb[j] + (int64_t)(rb + r) * rs[j]] = (double)T[m][j][r] + (double)acc[m][j][r];
    }
  }
}
template <int MT, int CT>
struct F_k_prop_split {
  static constexpr int NT = 64 * PS_WAVES, OCC = 1;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_prop_split_body<MT, CT>(b, g, a...);
  }
};
template <int MT, int CT>
__global__ __launch_bounds__(64 * PS_WAVES, 1) void k_prop_split(const u16* __restrict__ Vh, const u16* __restrict__ Vl,
                                                                 const u16* __restrict__ Dh, const u16* __restrict__ Dl,
                                                                 const double* src, double* dst, const double* weights,
                                                                 int N, int Nd, int na, int nb, int64_t offb,
                                                                 int64_t wstride, float sq, int nblk, int W) {
  k_prop_split_body<MT, CT>(blockIdx3(), gridDim3(), Vh, Vl, Dh, Dl, src, dst, weights, N, Nd, na, nb, offb, wstride, sq, nblk, W);
}

// V P -> the split [-P_im | P_re] chunks of k_taylor_h (used when the VHS ran in FP64)
__device__ __forceinline__ void k_v_split_body(const uint3 bid_, const uint3 gdim_, const double* P, u16* Vh, u16* Vl, const double* weights, int N, int Nq, int W) {
  const int nch = Nq >> 4;
  const int64_t per = (int64_t)nch * N * 32, total = per * W;
  for (int64_t e = (int64_t)bid_.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gdim_.x * blockDim.x) {
    const int w = (int)(e / per);
    if (weights[w] <= 1e-8) continue;
    const int64_t r = e - (int64_t)w * per;
    const int ch = (int)(r / ((int64_t)N * 32));
    const int rem = (int)(r - (int64_t)ch * N * 32), i = rem >> 5, pos = rem & 31;
    const int k = ch * 16 + (pos & 15);
    double x = 0.0;
    if (k < N) {
      const double* Pw = P + (int64_t)(2 * w) * N * N;
      x = pos < 16 ? -Pw[(int64_t)N * N + (int64_t)i * N + k] : Pw[(int64_t)i * N + k];
    }
    u16 h, l;
    split_bf16(x, h, l);
    Vh[e] = h;
    Vl[e] = l;
  }
}
struct F_k_v_split {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_v_split_body(b, g, a...);
  }
};
__global__ void k_v_split(const double* P, u16* Vh, u16* Vl, const double* weights, int N, int Nq, int W) {
  k_v_split_body(blockIdx3(), gridDim3(), P, Vh, Vl, weights, N, Nq, W);
}
void launch_v_split(const DevState& s, hipStream_t st) {
  const int64_t total = (int64_t)(s.Nq >> 4) * s.N * 32 * s.W;
  afq::glaunch<F_k_v_split>(k_v_split, dim3((unsigned)std::min<int64_t>(cdivu(total, 256), 65535)), dim3(256), 0, st, s.P,
                     s.Vh, s.Vl, s.weights, s.N, s.Nq, s.W);
}

// One-body factor in split BF16 with the identity kept exact: E = I + D with D = E - I
// small (|D| ~ dt/2 |h1'|), so E x = x + D x takes x in FP64 and only D x through three
// MFMA passes (hi*hi + hi*lo + lo*hi, FP32 accumulation).  D is split once per context
// (Dh/Dl, N rows of pitch Nd = N padded to 32, zero pads); x is split while staging.  Columns are the
// W * 2n real columns of one determinant of every walker (D is real).  mode 0:
// dst = E x and its split copy in t0b (the first Taylor term, columns from coloff of the
// ncolc propagated columns); mode 1: dst = E x.  Tile 32*MI rows x 256 columns.
template <int MI>
__device__ __forceinline__ void k_onebody_split_body(const uint3 bid_, const uint3 gdim_, const u16* Dh, const u16* Dl, const double* src, double* dst,
                                                       const double* weights, int N, int Nq, int Nd, int n, int W,
                                                       int64_t wstride, int64_t doff, int mode, u16* t0b, int coloff,
                                                       int ncolc, int gridx, int gridy) {
  constexpr int BM = 32 * MI, BN = 256;
  constexpr int AV = 2 * BM * 4, AVT = (AV + 511) / 512;
  __shared__ __attribute__((aligned(16))) u16 As[2][BM * TH_LDK];
  __shared__ __attribute__((aligned(16))) u16 Bs[2][BN * TH_LDK];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, 1, gridy);
  const int row0 = tl.y * BM, c0 = tl.x * BN;
  const int n2 = 2 * n, ncol = W * n2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 2, wn = wave & 3;
  // B: thread -> column c0 + (tid & 255), orbital groups of 8: (tid >> 8) and 2 + (tid >> 8)
  const int bc = c0 + (tid & 255);
  const double* bcol = nullptr;
  if (bc < ncol) {
    const int w = bc / n2;
    bcol = src + (int64_t)w * wstride + doff + (bc - w * n2);
  }
  uint4 ra[AVT];
  double rb[2][8];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int h = 0; h < AVT; ++h) {
      const int e = tid + 512 * h;
      ra[h] = uint4{0u, 0u, 0u, 0u};
      if (e < AV) {
        const int pl = e / (BM * 4), r = (e >> 2) - pl * BM, v = e & 3, i = row0 + r;
        if (i < N) ra[h] = *reinterpret_cast<const uint4*>((pl ? Dl : Dh) + (int64_t)i * Nd + k0 + 8 * v);
      }
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int kb = k0 + 8 * ((tid >> 8) + 2 * g);
#pragma unroll
      for (int t = 0; t < 8; ++t) rb[g][t] = (bcol && kb + t < N) ? bcol[(int64_t)(kb + t) * n2] : 0.0;
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int h = 0; h < AVT; ++h) {
      const int e = tid + 512 * h;
      if (e < AV) {
        const int pl = e / (BM * 4), r = (e >> 2) - pl * BM, v = e & 3;
        *reinterpret_cast<uint4*>(As[pl] + r * TH_LDK + 8 * v) = ra[h];
      }
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      unsigned hw[4], lw[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        u16 h0, l0, h1, l1;
        split_bf16(rb[g][2 * t], h0, l0);
        split_bf16(rb[g][2 * t + 1], h1, l1);
        hw[t] = (unsigned)h0 | ((unsigned)h1 << 16);
        lw[t] = (unsigned)l0 | ((unsigned)l1 << 16);
      }
      const int off = (tid & 255) * TH_LDK + 8 * ((tid >> 8) + 2 * g);
      *reinterpret_cast<uint4*>(Bs[0] + off) = uint4{hw[0], hw[1], hw[2], hw[3]};
      *reinterpret_cast<uint4*>(Bs[1] + off) = uint4{lw[0], lw[1], lw[2], lw[3]};
    }
  };
  f32x4 c[MI][4];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) c[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nst = Nd >> 5;
  fetch(0);
  for (int st = 0; st < nst; ++st) {
    stage();
    __syncthreads();
    if (st + 1 < nst) fetch((st + 1) * 32);
    const int koff = 8 * (lane >> 4);
    bf16x8 b[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        b[h][j] = *reinterpret_cast<const bf16x8*>(Bs[h] + (wn * 64 + j * 16 + (lane & 15)) * TH_LDK + koff);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(As[0] + (wm * 16 * MI + i * 16 + (lane & 15)) * TH_LDK + koff);
      const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(As[1] + (wm * 16 * MI + i * 16 + (lane & 15)) * TH_LDK + koff);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b[0][j], c[i][j], 0, 0, 0);
        c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b[1][j], c[i][j], 0, 0, 0);
        c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b[0][j], c[i][j], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  const int64_t plane = (int64_t)ncolc * Nq;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int col = c0 + wn * 64 + j * 16 + (lane & 15);
    if (col >= ncol) continue;
    const int w = col / n2, cc = col - w * n2;
    if (weights[w] <= 1e-8) continue;
    const int64_t base = (int64_t)w * wstride + doff + cc;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int rowb = row0 + wm * 16 * MI + i * 16 + 4 * (lane >> 4);
      if (rowb >= N) continue;
      float y[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = rowb + r;
        y[r] = 0.f;
        if (row < N) {
          const double v = src[base + (int64_t)row * n2] + (double)c[i][j][r];
          dst[base + (int64_t)row * n2] = v;
          y[r] = (float)v;
        }
      }
      if (mode == 0) {
        const int comp = cc & 1;
        const int64_t o = (int64_t)w * 4 * plane + 2 * comp * plane + ((int64_t)(rowb >> 4) * ncolc + coloff + (cc >> 1)) * 16 +
                          (rowb & 15);
        float yf[4] = {y[0], y[1], y[2], y[3]};
        uint2 oh, ol;
        split4_bf16(yf, oh, ol);
        *reinterpret_cast<uint2*>(t0b + o) = oh;
        *reinterpret_cast<uint2*>(t0b + o + plane) = ol;
      }
    }
  }
}
template <int MI>
struct F_k_onebody_split {
  static constexpr int NT = 512, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_onebody_split_body<MI>(b, g, a...);
  }
};
template <int MI>
__global__ __launch_bounds__(512) void k_onebody_split(const u16* Dh, const u16* Dl, const double* src, double* dst,
                                                       const double* weights, int N, int Nq, int Nd, int n, int W,
                                                       int64_t wstride, int64_t doff, int mode, u16* t0b, int coloff,
                                                       int ncolc, int gridx, int gridy) {
  k_onebody_split_body<MI>(blockIdx3(), gridDim3(), Dh, Dl, src, dst, weights, N, Nq, Nd, n, W, wstride, doff, mode, t0b, coloff, ncolc, gridx, gridy);
}

// D = E - I, split, N rows of pitch Nd (zero pads)
__device__ __forceinline__ void k_d_split_body(const uint3 bid_, const uint3 gdim_, const double* E, u16* Dh, u16* Dl, int N, int Nd) {
  const int64_t total = (int64_t)N * Nd;
  for (int64_t e = (int64_t)bid_.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gdim_.x * blockDim.x) {
    const int i = (int)(e / Nd), k = (int)(e - (int64_t)i * Nd);
    const double x = k < N ? E[(int64_t)i * N + k] - (i == k ? 1.0 : 0.0) : 0.0;
    u16 h, l;
    split_bf16(x, h, l);
    Dh[e] = h;
    Dl[e] = l;
  }
}
struct F_k_d_split {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_d_split_body(b, g, a...);
  }
};
__global__ void k_d_split(const double* E, u16* Dh, u16* Dl, int N, int Nd) {
  k_d_split_body(blockIdx3(), gridDim3(), E, Dh, Dl, N, Nd);
}
void launch_d_split(const DevState& s, hipStream_t st) {
  const int Nd = onebody_pitch(s.N);
  const int64_t total = (int64_t)s.N * Nd;
  afq::glaunch<F_k_d_split>(k_d_split, dim3((unsigned)std::min<int64_t>(cdivu(total, 256), 4096)), dim3(256), 0, st, s.E,
                     s.Dh, s.Dl, s.N, Nd);
}
template <int MI>
static void onebody_split(const DevState& s, const double* src, double* dst, int mode, hipStream_t st) {
  const int64_t ws = 2 * s.ms;
  const int ncolc = s.det_n[0] + (s.ndets_prop > 1 ? s.det_n[1] : 0);
  for (int d = 0; d < s.ndets_prop; ++d) {
    const int n = s.det_n[d];
    const int gx = (int)cdivu((int64_t)s.W * 2 * n, 256), gy = (int)cdivu(s.N, 32 * MI);
    afq::glaunch<F_k_onebody_split<MI>>((k_onebody_split<MI>), dim3(gx * gy), dim3(512), 0, st, s.Dh, s.Dl, src, dst, s.weights, s.N,
                       s.Nq, onebody_pitch(s.N), n, s.W, ws, 2 * s.det_off[d], mode, s.Ub[2], d ? s.det_n[0] : 0,
                       ncolc, gx, gy);
  }
}
static void launch_onebody_split(const DevState& s, const double* src, double* dst, int mode, hipStream_t st) {
  const int64_t p4 = (int64_t)cdivu(s.N, 128) * 128, p5 = (int64_t)cdivu(s.N, 160) * 160;
  if (p5 < p4) onebody_split<5>(s, src, dst, mode, st);
  else onebody_split<4>(s, src, dst, mode, st);
}

// ---- the fused split propagation (k_prop_split)
bool prop_fused_fits(const DevState& s) { return (s.N + 15) / 16 <= PS_WAVES * PS_MT_MAX; }
static bool prop_fused(const DevState& s) {
  if (s.prec_prop == AFQ_PREC_FP64 || !prop_fused_fits(s)) return false;
  return s.taylor_variant == 0 || s.taylor_variant == 3;
}
template <int MT, int CT>
static void prop_split_mc(const DevState& s, const double* src, double* dst, hipStream_t st) {
  const int na = s.det_n[0], nb = s.ndets_prop > 1 ? s.det_n[1] : 0;
  const int nblk = (int)cdivu(na + nb, 8 * CT);
  afq::glaunch<F_k_prop_split<MT, CT>>((k_prop_split<MT, CT>), dim3((unsigned)(nblk * s.W)), dim3(64 * PS_WAVES), 0, st, s.Vh, s.Vl,
                     s.Dh, s.Dl, src, dst, s.weights, s.N, onebody_pitch(s.N), na, nb, s.det_off[1], 2 * s.ms,
                     (float)sqrt(s.dt), nblk, s.W);
}
template <int MT>
static void prop_split_m(const DevState& s, int ct, const double* src, double* dst, hipStream_t st) {
  switch (ct) {
    case 1: prop_split_mc<MT, 1>(s, src, dst, st); break;
    case 2: prop_split_mc<MT, 2>(s, src, dst, st); break;
    case 3: prop_split_mc<MT, 3>(s, src, dst, st); break;
    default: prop_split_mc<MT, 4>(s, src, dst, st); break;
  }
}
// dst <- E (sum_{k<=5} V^k / k!) E src over the propagated columns (dst may be src)
static void launch_prop_fused(const DevState& s, const double* src, double* dst, hipStream_t st) {
  if (s.prec_vhs == AFQ_PREC_FP64) launch_v_split(s, st);
  // column tiles of 8 complex columns, at most 4 per block, spread evenly over the blocks
  // (at most 3, one block more per walker at N=300, 60+60, was slower: 10.4 against 9.3 ms)
  const int mt = (int)cdivu(cdivu(s.N, 16), PS_WAVES);
  const int ctot = (int)cdivu(s.det_n[0] + (s.ndets_prop > 1 ? s.det_n[1] : 0), 8);
  const int nblk = (int)cdivu(ctot, 4), ct = (int)cdivu(ctot, nblk);
  if (mt <= 1) prop_split_m<1>(s, ct, src, dst, st);
  else if (mt == 2) prop_split_m<2>(s, ct, src, dst, st);
  else prop_split_m<3>(s, ct, src, dst, st);
}
static void launch_taylor_split(const DevState& s, hipStream_t st);
static void launch_prop_split_to(const DevState& s, double* dst, hipStream_t st) {
  if (prop_fused(s)) {
    launch_prop_fused(s, s.psi, dst, st);
    return;
  }
  launch_onebody_split(s, s.psi, s.t0, 0, st);
  launch_taylor_split(s, st);
  launch_onebody_split(s, s.accb, dst, 1, st);
}

// the fused FP64 propagation (k_prop64) runs in launch_taylor
static bool prop64(const DevState& s) {
  return s.prec_prop == AFQ_PREC_FP64 && s.taylor_variant != 1 && s.taylor_variant != 2 && prop64_fits(s);
}
// psi <- E (sum_{k<=5} V^k / k!) E psi  for every live walker
bool prop_in_one(const DevState& s) { return prop64(s) || (s.prec_prop != AFQ_PREC_FP64 && prop_fused(s)); }
void launch_expmul_pre(const DevState& s, hipStream_t st) {
  if (prop64(s)) return;
  if (s.prec_prop != AFQ_PREC_FP64) {
    if (!prop_fused(s)) launch_onebody_split(s, s.psi, s.t0, 0, st);
    return;
  }
  const int64_t ws = 2 * s.ms;
  for (int d = 0; d < s.ndets_prop; ++d) {
    const int n = s.det_n[d];
    const int gx = (int)cdivu((int64_t)s.W * 2 * n, EX_BN), gy = (int)cdivu(s.N, EX_BM);
    const double* E = (s.uints && d == 1) ? s.E2 : s.E;  // spin d's propagator
    afq::glaunch<F_k_expmul>(k_expmul, dim3(gx * gy), dim3(256), 0, st, E, s.psi, s.t0, s.accb, s.weights, s.N,
                       n, s.W, ws, 2 * s.det_off[d], 0, gx, gy);
  }
}
template <int MI, int NI, int CPS = 1>   // two chunks per stage measured slower at N=300
static void taylor_split_steps(const DevState& s, hipStream_t st) {
  const int na = s.det_n[0], nb = s.ndets_prop > 1 ? s.det_n[1] : 0;
  const int gx = (int)cdivu(na + nb, 32 * NI), gy = (int)cdivu(s.N, 32 * MI);
  const u16* src = s.Ub[2];
  for (int p = 5; p >= 1; --p) {
    u16* dst = s.Ub[p & 1];
    afq::glaunch<F_k_taylor_h<MI, NI, CPS>>((k_taylor_h<MI, NI, CPS>), dim3(gx * gy * s.W), dim3(512), 0, st, s.Vh, s.Vl, src, dst, s.Ub[2],
                       s.t0, s.accb, s.weights, s.N, s.Nq, na, nb, s.det_off[1], 2 * s.ms,
                       (float)(sqrt(s.dt) / p), p == 1 ? 1 : 0, gx, gy, s.W);
    src = dst;
  }
}
// 128- or 160-row tiles (variant 1 / 2, or the one that pads N less), and 32, 64 or 128
// complex columns per tile
template <int MI>
static void taylor_split_cols(const DevState& s, hipStream_t st) {
  const int ncolc = s.det_n[0] + (s.ndets_prop > 1 ? s.det_n[1] : 0);
  if (ncolc <= 32) taylor_split_steps<MI, 1>(s, st);
  else if (ncolc <= 64) taylor_split_steps<MI, 2>(s, st);
  else taylor_split_steps<MI, 4>(s, st);
}
static void launch_taylor_split(const DevState& s, hipStream_t st) {
  if (s.prec_vhs == AFQ_PREC_FP64) launch_v_split(s, st);
  int v = s.taylor_variant;
  if (v != 1 && v != 2) {
    const int64_t p4 = (int64_t)cdivu(s.N, 128) * 128, p5 = (int64_t)cdivu(s.N, 160) * 160;
    v = p5 < p4 ? 2 : 1;
  }
  if (v == 2) taylor_split_cols<5>(s, st);
  else taylor_split_cols<4>(s, st);
}
// The Taylor products of the determinants listed: with a single determinant d the
// kernels see only its columns (a walker block offset to det d, no second part).
static void taylor_fp64(const DevState& s, const double* P, int dsel, hipStream_t st) {
  const int64_t ws = 2 * s.ms;
  const int na = dsel < 0 ? s.det_n[0] : s.det_n[dsel];
  const int nb = dsel < 0 && s.ndets_prop > 1 ? s.det_n[1] : 0;
  const int n2a = 2 * na, n2b = 2 * nb;
  const int64_t offb = 2 * s.det_off[1];
  const int64_t base = dsel > 0 ? 2 * s.det_off[dsel] : 0;
  const double sq = sqrt(s.dt);
  double* src = s.t0 + base;
  double* dst = s.t1 + base;
  double* acc = s.accb + base;
  const bool wide = (s.taylor_variant == 1 || s.taylor_variant == 2) ? s.taylor_variant == 2 : n2a + n2b > 128;
  for (int p = 1; p <= 5; ++p) {
    if (wide) {
      const int gx = (int)cdivu(na + nb, TY_BNC), gy = (int)cdivu(s.N, TY_BM);
      if (s.N % 2 == 0)
        afq::glaunch<F_k_taylor<true>>(k_taylor<true>, dim3(gx * gy * s.W), dim3(512), 0, st, P, src, dst, acc, s.weights,
                           s.N, na, nb, s.det_off[1], ws, sq / p, gx, gy, s.W);
      else
        afq::glaunch<F_k_taylor<false>>(k_taylor<false>, dim3(gx * gy * s.W), dim3(512), 0, st, P, src, dst, acc, s.weights,
                           s.N, na, nb, s.det_off[1], ws, sq / p, gx, gy, s.W);
    } else {
      const int gx = (int)cdivu(n2a + n2b, 128), gy = (int)cdivu(s.N, 64);
      afq::glaunch<F_k_vmul<64, 128, 2, 2>>((k_vmul<64, 128, 2, 2>), dim3(gx * gy * s.W), dim3(256), 0, st, P, src, dst, acc,
                         s.weights, s.N, s.T, n2a, n2b, offb, ws, sq, 1.0 / p, gx, gy, s.W);
    }
    double* t = src; src = dst; dst = t;
  }
}
void launch_taylor(const DevState& s, hipStream_t st) {
  if (prop64(s)) {
    launch_prop64(s, s.psi, st);
    return;
  }
  if (s.uints && s.prec_prop == AFQ_PREC_FP64) {
    // unrestricted integrals: each determinant with its own spin's V (DQMC/DQMCWalker.cpp:532-540)
    taylor_fp64(s, s.P, 0, st);
    taylor_fp64(s, s.P2, 1, st);
    return;
  }
  const int64_t ws = 2 * s.ms;
  const int n2a = 2 * s.det_n[0];
  const int n2b = s.ndets_prop > 1 ? 2 * s.det_n[1] : 0;
  const int64_t offb = 2 * s.det_off[1];
  const double sq = sqrt(s.dt);
  double* src = s.t0;
  double* dst = s.t1;
  const bool wide = (s.taylor_variant == 1 || s.taylor_variant == 2) ? s.taylor_variant == 2 : n2a + n2b > 128;
  const int na = s.det_n[0], nb = s.ndets_prop > 1 ? s.det_n[1] : 0;
  if (s.prec_prop != AFQ_PREC_FP64) {
    if (prop_fused(s)) launch_prop_fused(s, s.psi, s.psi, st);
    else launch_taylor_split(s, st);
    return;
  }
  for (int p = 1; p <= 5; ++p) {
    if (wide) {
      const int gx = (int)cdivu(na + nb, TY_BNC), gy = (int)cdivu(s.N, TY_BM);
      if (s.N % 2 == 0)
        afq::glaunch<F_k_taylor<true>>(k_taylor<true>, dim3(gx * gy * s.W), dim3(512), 0, st, s.P, src, dst, s.accb, s.weights,
                           s.N, na, nb, s.det_off[1], ws, sq / p, gx, gy, s.W);
      else
        afq::glaunch<F_k_taylor<false>>(k_taylor<false>, dim3(gx * gy * s.W), dim3(512), 0, st, s.P, src, dst, s.accb, s.weights,
                           s.N, na, nb, s.det_off[1], ws, sq / p, gx, gy, s.W);
    } else {
      const int gx = (int)cdivu(n2a + n2b, 128), gy = (int)cdivu(s.N, 64);
      afq::glaunch<F_k_vmul<64, 128, 2, 2>>((k_vmul<64, 128, 2, 2>), dim3(gx * gy * s.W), dim3(256), 0, st, s.P, src, dst, s.accb,
                         s.weights, s.N, s.T, n2a, n2b, offb, ws, sq, 1.0 / p, gx, gy, s.W);
    }
    double* t = src; src = dst; dst = t;
  }
}
// the closing FP64 one-body factor: dst <- E acc
static void expmul_post_to(const DevState& s, double* dst, hipStream_t st) {
  const int64_t ws = 2 * s.ms;
  for (int d = 0; d < s.ndets_prop; ++d) {
    const int n = s.det_n[d];
    const int gx = (int)cdivu((int64_t)s.W * 2 * n, EX_BN), gy = (int)cdivu(s.N, EX_BM);
    const double* E = (s.uints && d == 1) ? s.E2 : s.E;
    afq::glaunch<F_k_expmul>(k_expmul, dim3(gx * gy), dim3(256), 0, st, E, s.accb, dst, nullptr, s.weights,
                       s.N, n, s.W, ws, 2 * s.det_off[d], 1, gx, gy);
  }
}
void launch_expmul_post(const DevState& s, hipStream_t st) {
  if (prop64(s)) return;
  if (s.prec_prop == AFQ_PREC_FP64) expmul_post_to(s, s.psi, st);
  else if (!prop_fused(s)) launch_onebody_split(s, s.accb, s.psi, 1, st);
}
// The whole propagation (both one-body factors and the series) of the context's variant
// with the result in dst, which may be t1: the walkers stay as they are
void launch_propagate_to(const DevState& s, double* dst, hipStream_t st) {
  if (s.prec_prop != AFQ_PREC_FP64) {
    launch_prop_split_to(s, dst, st);
  } else if (prop64(s)) {
    launch_prop64(s, dst, st);
  } else {
    launch_expmul_pre(s, st);
    launch_taylor(s, st);
    expmul_post_to(s, dst, st);
  }
}
void launch_propagate(const DevState& s, hipStream_t st) {
  launch_expmul_pre(s, st);
  launch_taylor(s, st);
  launch_expmul_post(s, st);
}

// ------------------------------------------------------------------ Green's function
// The Green's function in three batched kernels (1 and 3 in afq_green.hip):
//  1. k_overlap: S = Phi_s^T psi for every walker of a slot as one GEMM over the
//     W * 2n real columns (FP64 MFMA), into Sg[w][slot] (64 x 128 doubles each);
//  2. k_invert: S^-1 and log det S per (walker, slot) by Gauss-Jordan elimination with
//     partial pivoting, the matrix held in registers (lane = row; one wave's columns, or
//     CPW q .. CPW q + CPW - 1 for wave q of several);
//  3. k_theta: theta = psi S^-1 (FP64 MFMA, S^-1 held in LDS) and the one-body
//     partial e1 = sum theta o (h1 Phi).
// In a propagation step 1-2 run before the weight update (the overlap ratio needs
// log det S of every propagated walker) and 3 after it, for the walkers still alive.
// one step of a wave maximum by a DPP move: a lane of the rows in RM takes the key of the lane
// CTRL names when that one is larger
template <int CTRL, int RM>
__device__ __forceinline__ unsigned dpp_max_step(unsigned v) {
  const unsigned o = (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, RM, 0xF, false);
  return max(v, o);
}

// x[0 .. CPW) are a wave's columns, in register slots that rotate: the wave that holds column k
// has it in slot 0, and its update moves every slot down one (the results simply go to the
// registers of the slot below) with column k's successor at the top, so that the step needs no
// register index and is not unrolled over k.
template <int CPW, bool MULTI>
__device__ __forceinline__ void k_invert_body(const uint3 bid_, const uint3 gdim_, GreenArgs a) {
  __shared__ cplx colb[2][GN_MAX];
  __shared__ cplx pvs[GN_MAX];
  __shared__ int pk[GN_MAX];
  const int w = bid_.x, si = bid_.y;
  const bool take = a.all || a.weights[w] > 1e-8;
  if (a.fresh && si == 0 && threadIdx.x == 0) a.fresh[w] = take ? 1 : 0;
  if (!take) return;
  const Slot sl = si == 0 ? a.s0 : a.s1;
  const int n = sl.n, tid = threadIdx.x, lane = tid & 63;
  const int q = !MULTI ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6);
  double* S = a.Sg + ((int64_t)w * a.nslots + si) * SG_MAT;
  cplx x[CPW];
#pragma unroll
  for (int j = 0; j < CPW; ++j) {
    const int col = CPW * q + j;
    x[j] = cplx{0.0, 0.0};
    if (lane < n && col < n) x[j] = cplx{S[lane * SG_LD + 2 * col], S[lane * SG_LD + 2 * col + 1]};
  }
  bool used = lane >= n;
  int myk = 0;
  for (int k = 0, o = 0, c = 0; k < n; ++k, ++c) {
    if (MULTI && c == CPW) {
      c = 0;
      ++o;
    }
    cplx f = x[0];
    if (MULTI) {
      if (q == o) colb[k & 1][lane] = x[0];
      __syncthreads();
      f = colb[k & 1][lane];
    }
    // pivot: the unused row of largest |f|^2, ties to the lower row.  |f|^2 >= 0, so its
    // high word orders like its value; its low 7 bits carry 64 - row (rows whose |f|^2 agree to
    // 2^-13 relative count as tied, and a pivot that close to the largest serves as well), and a
    // used row has key 0.  The maximum over the wave
    // by DPP moves (no LDS round trips): pairs, quads, half rows, rows, then rows 1 and 3
    // take rows 0 and 2, and row 3 takes row 1, so lane 63 ends with it.
    unsigned key = used ? 0u
                        : ((unsigned)__double2hiint(f.re * f.re + f.im * f.im) & ~0x7Fu) | (unsigned)(64 - lane);
    key = dpp_max_step<0xB1, 0xF>(key);    // quad_perm [1,0,3,2]
    key = dpp_max_step<0x4E, 0xF>(key);    // quad_perm [2,3,0,1]
    key = dpp_max_step<0x141, 0xF>(key);   // row_half_mirror
    key = dpp_max_step<0x140, 0xF>(key);   // row_mirror
    key = dpp_max_step<0x142, 0xA>(key);   // row_bcast:15 into rows 1 and 3
    key = dpp_max_step<0x143, 0xC>(key);   // row_bcast:31 into rows 2 and 3
    const int p = 64 - (int)(__builtin_amdgcn_readlane((int)key, 63) & 0x7F);
    const cplx pv{readlane_f64(f.re, p), readlane_f64(f.im, p)};
    // 1 / pv = conj(pv) / |pv|^2 (one division; the pivots of an overlap matrix are
    // far from the range where |pv|^2 would overflow or underflow)
    const double rn = 1.0 / (pv.re * pv.re + pv.im * pv.im);
    const cplx pinv{pv.re * rn, -pv.im * rn};
    if (lane == p) { used = true; myk = k; }
    if (tid == 0) {
      pk[k] = p;
      pvs[k] = pv;
    }
    // every other row minus (f_i / pv) times row p; row p itself keeps its scale
    // until the end (every row is divided by its own pivot after the last step, so
    // the update of a column is one complex multiply-add).  The stored column k
    // turns into column p of the inverse (in place): 1 in row p (divided by pv at
    // the end) and -f_i / pv elsewhere.
    cplx g = cmul(f, pinv);
    if (lane == p) g = cplx{0.0, 0.0};
    // four columns at a time, all broadcasts first: a use right behind its broadcast, and the
    // second FMA of an element right behind the first, would wait for it
    auto update = [&](auto from, auto to) {
#pragma unroll
      for (int j0 = 0; j0 < CPW; j0 += 4) {
        cplx xp[4], t[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (from(j0 + j) < CPW) xp[j] = cplx{readlane_f64(x[from(j0 + j)].re, p), readlane_f64(x[from(j0 + j)].im, p)};
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (from(j0 + j) < CPW) {
            const cplx v = x[from(j0 + j)];
            t[j] = cplx{v.re - g.re * xp[j].re, v.im - g.re * xp[j].im};
          }
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (from(j0 + j) < CPW) x[to(j0 + j)] = cplx{t[j].re + g.im * xp[j].im, t[j].im - g.im * xp[j].re};
      }
    };
    if (!MULTI || q == o) {
      update([](int j) { return j + 1; }, [](int j) { return j; });
      x[CPW - 1] = lane == p ? cplx{1.0, 0.0} : cplx{-g.re, -g.im};
    } else {
      update([](int j) { return j; }, [](int j) { return j; });
    }
  }
  // how far this wave's slots have rotated: slot j holds its column (j + rot) mod CPW
  const int rot = max(0, min(n - CPW * q, CPW));
  __syncthreads();
  if (lane < n) {
    // row p_k (this lane's, k = myk) divided by its pivot
    const cplx pm = pvs[myk];
    const double rn = 1.0 / (pm.re * pm.re + pm.im * pm.im);
    const cplx rinv{pm.re * rn, -pm.im * rn};
#pragma unroll
    for (int j = 0; j < CPW; ++j) x[j] = cmul(x[j], rinv);
  }
  // S^-1[k][p_j] = X[p_k][j]: lane p_k holds row myk, the slot of column j holds column p_j
  if (lane < n) {
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
      const int col = CPW * q + (j + rot < CPW ? j + rot : j + rot - CPW);
      if (col < n) {
        const int lc = pk[col];
        S[myk * SG_LD + 2 * lc] = x[j].re;
        S[myk * SG_LD + 2 * lc + 1] = x[j].im;
      }
    }
  }
  if (q == 0) {
    // det S = sign(k -> p_k) prod pivots
    cplx l = lane < n ? clog(pvs[lane]) : cplx{0.0, 0.0};
    const double ld_re = wave_sum(l.re);
    double ld_im = wave_sum(l.im);
    // the sign by the inversions of k -> p_k, each lane counting its own
    int inv = 0;
    const int mine = lane < n ? pk[lane] : 0;
    for (int k = 0; k + 1 < n; ++k) inv += lane > k && lane < n && pk[k] > mine ? 1 : 0;
    const unsigned long long odd = __ballot(inv & 1);
    if (__popcll(odd) & 1) ld_im += M_PI;
    if (lane == 0) {
      a.logdet[2 * ((int64_t)w * a.nslots + si)] = ld_re;
      a.logdet[2 * ((int64_t)w * a.nslots + si) + 1] = ld_im;
    }
  }
}
// waves a SIMD holds: 4 CPW registers for the columns and about 50 more
constexpr int inv_occ(int cpw) { return cpw <= 12 ? 4 : cpw <= 24 ? 3 : 2; }
template <int CPW, bool MULTI>
struct F_k_invert {
  static constexpr int NT = MULTI ? 256 : 64, OCC = inv_occ(CPW);
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_invert_body<CPW, MULTI>(b, g, a...);
  }
};
template <int CPW, bool MULTI>
__global__ __launch_bounds__(MULTI ? 256 : 64, inv_occ(CPW)) void k_invert(GreenArgs a) {
  k_invert_body<CPW, MULTI>(blockIdx3(), gridDim3(), a);
}

// Bound by VALU issue, of which a step's pivot search and division are about as much as the
// update of 8 columns, and with few matrices by a step's latency.  So one wave takes a whole
// matrix up to n = 32, without barriers, where there are more matrices than half the SIMDs (2048
// of n = 20: 48 us, three waves of 8 columns 58; 24 systems of n = 4 to 24, 256 walkers: 161 us
// against 213), and with fewer several waves share one (32 of n = 20: 17 us, one wave 21).  Past n = 32 four waves
// of 16 columns: 1.02 ms for 8192 matrices of n = 60 and 90 us for 512 (two of 32: 1.01 and 140).
static void launch_invert(const GreenArgs& a, hipStream_t st) {
  const int nmax = std::max(a.s0.n, a.nslots > 1 ? a.s1.n : 0);
  const dim3 grid(a.W, a.nslots);
  const bool few = (int64_t)a.W * a.nslots <= 512 && !g_recorder;   // a grouped launch fills the chip
#define AFQ_INV(CPW, MULTI) \
  afq::glaunch<F_k_invert<CPW, MULTI>>((k_invert<CPW, MULTI>), grid, dim3(MULTI ? 64 * cdivu(nmax, CPW) : 64), 0, st, a)
  if (nmax > 32) AFQ_INV(16, true);
  else if (few && nmax > 16) AFQ_INV(8, true);
  else if (few) AFQ_INV(4, true);
  else if (nmax <= 8) AFQ_INV(8, false);
  else if (nmax <= 12) AFQ_INV(12, false);
  else if (nmax <= 16) AFQ_INV(16, false);
  else if (nmax <= 20) AFQ_INV(20, false);
  else if (nmax <= 24) AFQ_INV(24, false);
  else AFQ_INV(32, false);
#undef AFQ_INV
}

static GreenArgs green_args(const DevState& s, bool all) {
  GreenArgs a;
  a.psi = s.psi; a.theta = s.theta; a.logdet = s.logdet; a.e1 = s.e1; a.weights = s.weights; a.Sg = s.Sg;
  a.phi0 = s.phi[0]; a.phi1 = s.phi[1]; a.hphi0 = s.hphi[0]; a.hphi1 = s.hphi[1];
  a.ms = s.ms; a.Ktot = s.Ktot; a.det_off0 = s.det_off[0]; a.det_off1 = s.det_off[1];
  a.N = s.N; a.nslots = s.nslots; a.W = s.W; a.s0 = s.slot[0]; a.s1 = s.slot[s.nslots > 1 ? 1 : 0]; a.all = all;
  return a;
}
// S = Phi^T psi and S^-1 / log det S of the walkers above the propagation threshold
// (every walker with all), marking them in s.gfresh
void launch_green_pre(const DevState& s, bool all, hipStream_t st) {
  s.tb_live = false;
  s.tb_post = false;
  GreenArgs a = green_args(s, all);
  a.fresh = s.gfresh;
  launch_overlap(a, st);
  launch_invert(a, st);
}
// theta = psi S^-1 (and e1) after the weight update, for the walkers launch_green_pre
// took that are still alive: the others are never read before the next step recomputes
// them (a walker of weight zero is neither measured nor given a force bias, and the comb
// replaces it)
void launch_theta_post(const DevState& s, hipStream_t st) {
  GreenArgs a = green_args(s, false);
  a.fresh = s.gfresh;
  a.post = 1;
  if (s.prec_fb != AFQ_PREC_FP64 && s.Tb_hi) {
    // the split force bias that follows reads these walkers' Tb from here
    a.tbh = s.Tb_hi;
    a.tbl = s.Tb_lo;
    a.Np = s.Np;
    a.ctot = s.ctot;
  }
  launch_theta(a, st);
  s.tb_post = a.tbh != nullptr;
}
void launch_green(const DevState& s, bool all, hipStream_t st) {
  s.tb_live = false;
  s.tb_post = false;
  const GreenArgs a = green_args(s, all);
  launch_overlap(a, st);
  launch_invert(a, st);
  launch_theta(a, st);
}

// ------------------------------------------------------------------ weights
// phaseless factor of DQMC/DQMCWalker.cpp:495-502 and the driver's update/cap
// (DQMC/MixedEstimator.cpp:461-468), with log overlaps.
__device__ __forceinline__ void k_weight_body(const uint3 bid_, const uint3 gdim_, double* weights, double* factors, double* logO, const double* logdet,
                         const double* sft, int W, int nslots, int m0, int m1, double dt, double eshift,
                         double pc_re, double cap, unsigned long long* ncap, int update,
                         const double* eshift_dev) {
  const int w = bid_.x * blockDim.x + threadIdx.x;
  // ncap[1] counts the walkers this step propagates (weight > 1e-8 at its start)
  const bool prop = w < W && weights[w] > 1e-8;
  const unsigned long long pm = __ballot(prop);
  if ((threadIdx.x & 63) == 0 && pm) atomicAdd(ncap + 1, (unsigned long long)__popcll(pm));
  if (w >= W) return;
  if (eshift_dev) eshift = *eshift_dev;
  double f = 1.0;
  if (prop) {
    double lo_re = m0 * logdet[2 * (int64_t)w * nslots], lo_im = m0 * logdet[2 * (int64_t)w * nslots + 1];
    if (nslots > 1) {
      lo_re += m1 * logdet[2 * ((int64_t)w * nslots + 1)];
      lo_im += m1 * logdet[2 * ((int64_t)w * nslots + 1) + 1];
    }
    const double dre = lo_re - logO[2 * w], dim = lo_im - logO[2 * w + 1];
    const double sq = sqrt(dt);
    const double zre = -sq * sft[4 * w] + sft[4 * w + 2] + dt * (eshift + pc_re) + dre;
    const double zth = -sq * sft[4 * w + 1] + dim;
    f = exp(zre) * cos(zth);
    if (!(f >= 1.e-3) || f > 100.) f = 0.0;
    if (update) weights[w] *= f;
    logO[2 * w] = lo_re;
    logO[2 * w + 1] = lo_im;
  }
  if (update && weights[w] > cap) {
    weights[w] = 0.0;
    atomicAdd(ncap, 1ull);
  }
  factors[w] = f;
}
struct F_k_weight {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_weight_body(b, g, a...);
  }
};
__global__ void k_weight(double* weights, double* factors, double* logO, const double* logdet,
                         const double* sft, int W, int nslots, int m0, int m1, double dt, double eshift,
                         double pc_re, double cap, unsigned long long* ncap, int update,
                         const double* eshift_dev) {
  k_weight_body(blockIdx3(), gridDim3(), weights, factors, logO, logdet, sft, W, nslots, m0, m1, dt, eshift, pc_re, cap, ncap, update, eshift_dev);
}

void launch_weight(const DevState& s, double eshift, bool update, hipStream_t st) {
  afq::glaunch<F_k_weight>(k_weight, dim3(cdivu(s.W, 256)), dim3(256), 0, st, s.weights, s.factors, s.logO,
                     s.logdet, s.sft, s.W, s.nslots, s.slot[0].mult, s.nslots > 1 ? s.slot[1].mult : 0,
                     s.dt, eshift, s.prop_const_re, s.weight_cap, s.ncap, (int)update, s.d_eshift);
}

__device__ __forceinline__ void k_logO_body(const uint3 bid_, const uint3 gdim_, double* logO, const double* logdet, int W, int nslots, int m0, int m1) {
  const int w = bid_.x * blockDim.x + threadIdx.x;
  if (w >= W) return;
  double re = m0 * logdet[2 * (int64_t)w * nslots], im = m0 * logdet[2 * (int64_t)w * nslots + 1];
  if (nslots > 1) {
    re += m1 * logdet[2 * ((int64_t)w * nslots + 1)];
    im += m1 * logdet[2 * ((int64_t)w * nslots + 1) + 1];
  }
  logO[2 * w] = re;
  logO[2 * w + 1] = im;
}
struct F_k_logO {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_logO_body(b, g, a...);
  }
};
__global__ void k_logO(double* logO, const double* logdet, int W, int nslots, int m0, int m1) {
  k_logO_body(blockIdx3(), gridDim3(), logO, logdet, W, nslots, m0, m1);
}

void launch_logO_from_logdet(const DevState& s, hipStream_t st) {
  afq::glaunch<F_k_logO>(k_logO, dim3(cdivu(s.W, 256)), dim3(256), 0, st, s.logO, s.logdet, s.W, s.nslots,
                     s.slot[0].mult, s.nslots > 1 ? s.slot[1].mult : 0);
}

// ------------------------------------------------------------------ Householder QR
// Thin Householder QR with Eigen's conventions (eigen/Eigen/src/Householder/Householder.h:63-92,
// eigen/Eigen/src/QR/HouseholderQR.h:267-297); psi_d := Q, logO -= log prod diag R
// (DQMC/DQMCWalker.cpp:295-326).  One workgroup per walker, both determinants.
__device__ __forceinline__ void k_qr_body(const uint3 bid_, const uint3 gdim_, double* psi, double* Qs, double* logO, const double* weights, int N,
                                            int ndets, int na, int nb, int64_t offb, int64_t ms, int rhf_walker) {
  __shared__ cplx tau[GN_MAX];
  __shared__ cplx tmp[GN_MAX];
  __shared__ double red[16];
  __shared__ double sbeta;
  __shared__ cplx sden;
  __shared__ int szero;
  const int w = bid_.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwv = blockDim.x >> 6;
  if (weights[w] == 0.0) return;   // weight zero: never read again before the comb replaces it
  double lf_re = 0.0, lf_im = 0.0;
  for (int d = 0; d < ndets; ++d) {
    const int n = d == 0 ? na : nb;
    cplx* A = reinterpret_cast<cplx*>(psi + 2 * ((int64_t)w * ms + (d == 0 ? 0 : offb)));
    cplx* Q = reinterpret_cast<cplx*>(Qs + 2 * ((int64_t)w * ms + (d == 0 ? 0 : offb)));
    for (int k = 0; k < n; ++k) {
      double t = 0.0;
      for (int i = k + 1 + tid; i < N; i += blockDim.x) {
        const cplx x = A[(int64_t)i * n + k];
        t += x.re * x.re + x.im * x.im;
      }
      const double tail = block_sum(t, red);
      if (tid == 0) {
        const cplx c0 = A[(int64_t)k * n + k];
        if (tail <= DBL_MIN && c0.im * c0.im <= DBL_MIN) {
          tau[k] = cplx{0.0, 0.0};
          sbeta = c0.re;
          szero = 1;
        } else {
          double beta = sqrt(c0.re * c0.re + c0.im * c0.im + tail);
          if (c0.re >= 0.0) beta = -beta;
          sbeta = beta;
          sden = cplx{c0.re - beta, c0.im};
          const cplx tt = cdiv(cplx{beta - c0.re, -c0.im}, cplx{beta, 0.0});
          tau[k] = cplx{tt.re, -tt.im};
          szero = 0;
        }
      }
      __syncthreads();
      const double beta = sbeta;
      for (int i = k + 1 + tid; i < N; i += blockDim.x)
        A[(int64_t)i * n + k] = szero ? cplx{0.0, 0.0} : cdiv(A[(int64_t)i * n + k], sden);
      if (tid == 0) {
        A[(int64_t)k * n + k] = cplx{beta, 0.0};
        lf_re += log(fabs(beta));
        if (beta < 0.0) lf_im += M_PI;
      }
      __syncthreads();
      // tmp_j = A(k,j) + sum_{i>k} conj(v_i) A(i,j), j > k
      for (int j = k + 1 + wave; j < n; j += nwv) {
        double sr = 0.0, si = 0.0;
        for (int i = k + 1 + lane; i < N; i += 64) {
          const cplx v = A[(int64_t)i * n + k], x = A[(int64_t)i * n + j];
          sr += v.re * x.re + v.im * x.im;
          si += v.re * x.im - v.im * x.re;
        }
        sr = wave_sum(sr);
        si = wave_sum(si);
        if (lane == 0) {
          const cplx akj = A[(int64_t)k * n + j];
          tmp[j] = cplx{akj.re + sr, akj.im + si};
        }
      }
      __syncthreads();
      const cplx tk = tau[k];
      const int nc = n - k - 1;
      for (int e = tid; e < (N - k) * nc; e += blockDim.x) {
        const int i = k + e / nc, j = k + 1 + e % nc;
        const cplx v = i == k ? cplx{1.0, 0.0} : A[(int64_t)i * n + k];
        const cplx u = cmul(tk, cmul(v, tmp[j]));
        A[(int64_t)i * n + j] = csub(A[(int64_t)i * n + j], u);
      }
      __syncthreads();
    }
    // Q = H_0^* ... H_{n-1}^* [I;0],  H_k^* = I - conj(tau_k) v v^*
    for (int e = tid; e < N * n; e += blockDim.x) {
      const int i = e / n, j = e - i * n;
      Q[e] = cplx{i == j ? 1.0 : 0.0, 0.0};
    }
    __syncthreads();
    for (int k = n - 1; k >= 0; --k) {
      const cplx tk = cplx{tau[k].re, -tau[k].im};
      for (int j = k + wave; j < n; j += nwv) {
        double sr = 0.0, si = 0.0;
        for (int i = k + 1 + lane; i < N; i += 64) {
          const cplx v = A[(int64_t)i * n + k], x = Q[(int64_t)i * n + j];
          sr += v.re * x.re + v.im * x.im;
          si += v.re * x.im - v.im * x.re;
        }
        sr = wave_sum(sr);
        si = wave_sum(si);
        if (lane == 0) {
          const cplx qkj = Q[(int64_t)k * n + j];
          tmp[j] = cplx{qkj.re + sr, qkj.im + si};
        }
      }
      __syncthreads();
      const int nc = n - k;
      for (int e = tid; e < (N - k) * nc; e += blockDim.x) {
        const int i = k + e / nc, j = k + e % nc;
        const cplx v = i == k ? cplx{1.0, 0.0} : A[(int64_t)i * n + k];
        Q[(int64_t)i * n + j] = csub(Q[(int64_t)i * n + j], cmul(tk, cmul(v, tmp[j])));
      }
      __syncthreads();
    }
    for (int e = tid; e < N * n; e += blockDim.x) A[e] = Q[e];
    __syncthreads();
  }
  if (tid == 0) {
    const double m = rhf_walker ? 2.0 : 1.0;
    logO[2 * w] -= m * lf_re;
    logO[2 * w + 1] -= m * lf_im;
  }
}
struct F_k_qr {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_qr_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_qr(double* psi, double* Qs, double* logO, const double* weights, int N,
                                            int ndets, int na, int nb, int64_t offb, int64_t ms, int rhf_walker) {
  k_qr_body(blockIdx3(), gridDim3(), psi, Qs, logO, weights, N, ndets, na, nb, offb, ms, rhf_walker);
}

// k_qr_cols for N <= 320 and n <= 64, k_qr otherwise
void launch_qr(const DevState& s, hipStream_t st) {
  if (launch_qr_cols(s, st)) return;
  afq::glaunch<F_k_qr>(k_qr, dim3(s.W), dim3(256), 0, st, s.psi, s.t0, s.logO, s.weights, s.N, s.ndets_prop,
                     s.det_n[0], s.det_n[1], s.det_off[1], s.ms, (int)s.walker_rhf);
}

// ------------------------------------------------------------------ exchange
// Epilogue shared by the FP64 and BF16 exchange kernels.  F holds one g-block of
// the tile's f = R_g theta for wt walkers: f_w(i, j) at F[i*LDF + 2n*w + 2j] (re, im).
// The 256 threads split into wt groups of tpw (a power of two) and each group sums
// f_ij f_ji over its walker's n^2 pairs; LDF is odd so the transposed reads f_ji
// of consecutive threads fall in different banks.
struct XPairs {
  int tpw, wl, lt;
  __device__ XPairs(int wt, int nthreads = 256) {
    int t = nthreads / wt, p = 1;
    while (2 * p <= t) p *= 2;
    tpw = p;
    wl = threadIdx.x / tpw;
    lt = threadIdx.x - wl * tpw;
  }
  template <class T>
  __device__ __forceinline__ void add(const T* F, int LDF, int n, int wt, double& accr, double& acci) const {
    if (wl >= wt) return;
    const T* Fw = F + wl * 2 * n;
    const int step_i = tpw / n, step_j = tpw - step_i * n;
    int i = lt / n, j = lt - i * n;
    for (; i < n;) {
      const double ar = Fw[i * LDF + 2 * j], ai = Fw[i * LDF + 2 * j + 1];
      const double br = Fw[j * LDF + 2 * i], bi = Fw[j * LDF + 2 * i + 1];
      accr += ar * br - ai * bi;
      acci += ar * bi + ai * br;
      i += step_i;
      j += step_j;
      if (j >= n) { j -= n; ++i; }
    }
  }
  // group sums; returns true on the thread that holds its walker's total
  __device__ __forceinline__ bool finish(double& accr, double& acci, double* red) const {
    const int gsz = tpw < 64 ? tpw : 64;
    for (int off = gsz / 2; off > 0; off >>= 1) {
      accr += __shfl_xor(accr, off, 64);
      acci += __shfl_xor(acci, off, 64);
    }
    if (tpw > 64) {
      const int wave = threadIdx.x >> 6;
      if ((threadIdx.x & 63) == 0) { red[2 * wave] = accr; red[2 * wave + 1] = acci; }
      __syncthreads();
      if (lt == 0) {
        accr = acci = 0.0;
        for (int q = wave; q < wave + tpw / 64; ++q) { accr += red[2 * q]; acci += red[2 * q + 1]; }
      }
    }
    return lt == 0;
  }
};

// The same pair sum over a whole tile of f held in LDS as FP32 at once: rows gl*n + i
// (g-block gl of the tile), columns wl*2n + 2j + {re, im} (walker wl), an even row
// pitch so (re, im) reads are 8-byte.  A walker's tpw threads split its gt*n rows
// ("units"); tpu threads share a unit and stride its n columns.  Per unit the inner
// sum runs in ACC (float for the one-pass surrogate, double otherwise).
template <class ACC>
struct XPairsF : XPairs {
  __device__ XPairsF(int wt) : XPairs(wt) {}
  __device__ __forceinline__ void add(const float* F, int LDF, int n, int gt, int wt, double& accr,
                                      double& acci) const {
    if (wl >= wt) return;
    const float* Fw = F + wl * 2 * n;
    const int units = gt * n;
    int tpu = 1;
    while (tpu * 2 * units <= tpw) tpu *= 2;
    const int ustep = tpw / tpu, j0 = lt & (tpu - 1);
    for (int u = lt / tpu; u < units; u += ustep) {
      const int gl = u / n, i = u - gl * n;
      const float* ri = Fw + u * LDF;
      const float* cj = Fw + gl * n * LDF + 2 * i;
      ACC sr = 0, si = 0;
      for (int j = j0; j < n; j += tpu) {
        const float2 a = *reinterpret_cast<const float2*>(ri + 2 * j);
        const float2 b = *reinterpret_cast<const float2*>(cj + j * LDF);
        sr += (ACC)a.x * (ACC)b.x - (ACC)a.y * (ACC)b.y;
        si += (ACC)a.x * (ACC)b.y + (ACC)a.y * (ACC)b.x;
      }
      accr += (double)sr;
      acci += (double)si;
    }
  }
};

constexpr int XC_BM = 128, XC_BN = 128;
int exchange_tile_g(int n) { return (n >= 1 && n <= XC_BN / 2) ? XC_BM / n : 0; }
int exchange_tile_w(int n) { return (n >= 1 && n <= XC_BN / 2) ? XC_BN / (2 * n) : 0; }

struct XcA {  // A((g,i), k) = R_{s,g}(i, k) = R[g][koff + k*n + i]
  const double* R; int64_t Ktot, koff; int n, gt, g0, GE, N;
  __device__ double operator()(int r, int k) const {
    const int gl = r / n, i = r - gl * n, g = g0 + gl;
    if (gl >= gt || g >= GE || k >= N) return 0.0;
    return R[(int64_t)g * Ktot + koff + (int64_t)k * n + i];
  }
};
struct XcB {  // B(k, (w,j,c)) = theta_s[w][k][j][c]
  const double* th; const int* sel; int64_t Ktot, koff; int n, wt, w0, nw, N;
  __device__ double operator()(int k, int c) const {
    const int n2 = 2 * n, wl = c / n2, cc = c - wl * n2;
    if (wl >= wt || w0 + wl >= nw || k >= N) return 0.0;
    const int w = sel ? sel[w0 + wl] : w0 + wl;
    return th[(int64_t)w * 2 * Ktot + 2 * koff + (int64_t)k * n2 + cc];
  }
};

// Xp[s][w][gtile] = sum_{g in tile} sum_ij f_ij f_ji,  f = R_{s,g} theta_s.
// The output tile is reduced one g-block at a time: its n rows are staged in
// LDS and summed by XPairs, so f never leaves the workgroup.
// With nsel_dev the selection's length is read from the device (nw is then only the
// bound the grid was sized for) and tiles past it exit.
__device__ __forceinline__ void k_exchange_body(const uint3 bid_, const uint3 gdim_, const double* R, const double* theta, const int* sel,
                                                     const int* nsel_dev, double* Xp, int N, int GE, int nw, int W,
                                                     int64_t Ktot, Slot s0, Slot s1, int ngt, int gridx, int gridy,
                                                     int gridz) {
  using Eng = MmaF64<XC_BM, XC_BN, 2, 2, true, true>;
  constexpr int LDF = XC_BN + 1;
  constexpr int FT = (XC_BN / 2) * LDF;
  constexpr int LDSN = Eng::LDS_DOUBLES > FT ? Eng::LDS_DOUBLES : FT;
  __shared__ double lds[LDSN];
  __shared__ double red[8];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, gridz, 8);
  const Slot sl = tl.z == 0 ? s0 : s1;
  const int n = sl.n, gt = XC_BM / n, wt = XC_BN / (2 * n);
  const int g0 = tl.x * gt, w0 = tl.y * wt;
  if (nsel_dev) nw = *nsel_dev;
  if (w0 >= nw) return;
  Eng e;
  e.run(XcA{R, Ktot, sl.koff, n, gt, g0, GE, N}, XcB{theta, sel, Ktot, sl.koff, n, wt, w0, nw, N}, N, lds);
  const XPairs xp(wt);
  double accr = 0.0, acci = 0.0;
  for (int gl = 0; gl < gt; ++gl) {
    if (g0 + gl >= GE) break;
    e.store([&](int r, int c, double v) {
      const int rr = r - gl * n;
      if (rr >= 0 && rr < n) lds[rr * LDF + c] = v;
    });
    __syncthreads();
    xp.add(lds, LDF, n, wt, accr, acci);
    __syncthreads();
  }
  if (xp.finish(accr, acci, red) && xp.wl < wt && w0 + xp.wl < nw) {
    const int w = sel ? sel[w0 + xp.wl] : w0 + xp.wl;
    double* o = Xp + 2 * (((int64_t)tl.z * W + w) * ngt + tl.x);
    o[0] = accr;
    o[1] = acci;
  }
}
struct F_k_exchange {
  static constexpr int NT = 256, OCC = 2;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_exchange_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256, 2) void k_exchange(const double* R, const double* theta, const int* sel,
                                                     const int* nsel_dev, double* Xp, int N, int GE, int nw, int W,
                                                     int64_t Ktot, Slot s0, Slot s1, int ngt, int gridx, int gridy,
                                                     int gridz) {
  k_exchange_body(blockIdx3(), gridDim3(), R, theta, sel, nsel_dev, Xp, N, GE, nw, W, Ktot, s0, s1, ngt, gridx, gridy, gridz);
}

// k_exchange on the pointer-loader engine (MmaF64P: double-buffered stages, no index
// arithmetic per element): 128 x 128 tiles over 4 (WN = 2) or 8 waves (WN = 4).
template <int WN>
__device__ __forceinline__ void k_exchange2_body(const uint3 bid_, const uint3 gdim_, const double* R, const double* theta, const int* sel,
                                                          const int* nsel_dev, double* Xp, int N, int GE, int nw,
                                                          int W, int64_t Ktot, Slot s0, Slot s1, int ngt, int gridx,
                                                          int gridy, int gridz) {
  using Eng = MmaF64P<XC_BM, XC_BN, 2, WN>;
  constexpr int NTH = 128 * WN;
  constexpr int LDF = XC_BN + 1;
  constexpr int FT = (XC_BN / 2) * LDF;
  constexpr int LDSN = Eng::LDS_DOUBLES > FT ? Eng::LDS_DOUBLES : FT;
  __shared__ double lds[LDSN];
  __shared__ double red[16];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, gridz, 8);
  const Slot sl = tl.z == 0 ? s0 : s1;
  const int n = sl.n, gt = XC_BM / n, wt = XC_BN / (2 * n);
  const int g0 = tl.x * gt, w0 = tl.y * wt;
  if (nsel_dev) nw = *nsel_dev;
  if (w0 >= nw) return;
  Eng e;
  e.run(
      [&](int r) -> const double* {   // A row (g, i): R_{s,g}(i, k) at R[g][koff + k n + i]
        const int gl = r / n, i = r - gl * n, g = g0 + gl;
        return (gl < gt && g < GE) ? R + (int64_t)g * Ktot + sl.koff + i : nullptr;
      },
      [&](int c) -> const double* {   // B column (w, j, re/im): theta_s[w][k][j][c]
        const int wl = c / (2 * n), cc = c - wl * 2 * n;
        if (wl >= wt || w0 + wl >= nw) return nullptr;
        const int w = sel ? sel[w0 + wl] : w0 + wl;
        return theta + (int64_t)w * 2 * Ktot + 2 * sl.koff + cc;
      },
      n, 2 * n, N, lds);
  const XPairs xp(wt, NTH);
  double accr = 0.0, acci = 0.0;
  for (int gl = 0; gl < gt; ++gl) {
    if (g0 + gl >= GE) break;
    e.store([&](int r, int c, double v) {
      const int rr = r - gl * n;
      if (rr >= 0 && rr < n) lds[rr * LDF + c] = v;
    });
    __syncthreads();
    xp.add(lds, LDF, n, wt, accr, acci);
    __syncthreads();
  }
  if (xp.finish(accr, acci, red) && xp.wl < wt && w0 + xp.wl < nw) {
    const int w = sel ? sel[w0 + xp.wl] : w0 + xp.wl;
    double* o = Xp + 2 * (((int64_t)tl.z * W + w) * ngt + tl.x);
    o[0] = accr;
    o[1] = acci;
  }
}
template <int WN>
struct F_k_exchange2 {
  static constexpr int NT = 128 * WN, OCC = 2;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_exchange2_body<WN>(b, g, a...);
  }
};
template <int WN>
__global__ __launch_bounds__(128 * WN, 2) void k_exchange2(const double* R, const double* theta, const int* sel,
                                                          const int* nsel_dev, double* Xp, int N, int GE, int nw,
                                                          int W, int64_t Ktot, Slot s0, Slot s1, int ngt, int gridx,
                                                          int gridy, int gridz) {
  k_exchange2_body<WN>(blockIdx3(), gridDim3(), R, theta, sel, nsel_dev, Xp, N, GE, nw, W, Ktot, s0, s1, ngt, gridx, gridy, gridz);
}

void launch_exchange(const DevState& s, const int* sel, int nsel, hipStream_t st, const int* nsel_dev) {
  // the slots [z0, z0 + nz) in one grid (slots of one size share a tile shape)
  auto go = [&](int z0, int nz) {
    const Slot a = s.slot[z0], b = s.slot[z0 + nz - 1];
    double* xp = s.Xp + 2 * (int64_t)z0 * s.W * s.ngt_cap;
    if (s.xc64_variant == 0 && a.n >= X64_NMIN) {
      launch_exchange64(s, sel, nsel, nsel_dev, xp, a, b, nz, st);
      return;
    }
    const int gt = exchange_tile_g(a.n), wt = exchange_tile_w(a.n);
    const int ngt = (int)cdivu(s.GE, gt), gy = (int)cdivu(nsel, wt);
    const dim3 grid(ngt * gy * nz);
    if (s.xc64_variant == 1)
      afq::glaunch<F_k_exchange>(k_exchange, grid, dim3(256), 0, st, s.R, s.theta, sel, nsel_dev, xp, s.N, s.GE, nsel, s.W,
                                 s.Ktot, a, b, s.ngt_cap, ngt, gy, nz);
    else if (s.xc64_variant == 2)
      afq::glaunch<F_k_exchange2<2>>((k_exchange2<2>), grid, dim3(256), 0, st, s.R, s.theta, sel, nsel_dev, xp, s.N, s.GE, nsel,
                                     s.W, s.Ktot, a, b, s.ngt_cap, ngt, gy, nz);
    else   // up to 3 electrons, eight waves: n = 1, 2, 3 at N = 50, G = 200, 1024 walkers 139, 78 and 83 us (four waves 163,
           // 90 and 85); n = 3 at N = 100, G = 400, 4096 walkers 656 us (731), at N = 12, G = 48, 256 walkers 51 (62)
      afq::glaunch<F_k_exchange2<4>>((k_exchange2<4>), grid, dim3(512), 0, st, s.R, s.theta, sel, nsel_dev, xp, s.N, s.GE, nsel,
                                     s.W, s.Ktot, a, b, s.ngt_cap, ngt, gy, nz);
  };
  if (s.nslots == 1 || s.slot[1].n == s.slot[0].n) {
    go(0, s.nslots);
  } else {
    go(0, 1);
    go(1, 1);
  }
}

// ------------------------------------------------------------------ mixed-precision exchange
// bf16 hi/lo copies, K (orbital) contiguous and padded to Np:
//   Rb[c][slot][g][i][Np]          from R[g][koff_s + k*n_s + i]
//   Tb[c][w][re/im][slot][j][Np]                   from theta_s[w][k][j][re/im]
__device__ __forceinline__ void k_rsplit_body(const uint3 bid_, const uint3 gdim_, const double* R, u16* hi, u16* lo, int N, int Np, int G, int64_t Ktot, int64_t koff,
                         int n, int64_t dst_off) {
  const int64_t total = (int64_t)G * n * Np;
  for (int64_t e = (int64_t)bid_.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gdim_.x * blockDim.x) {
    const int k = (int)(e % Np);
    const int64_t gi = e / Np;
    const int i = (int)(gi % n), g = (int)(gi / n);
    const double x = k < N ? R[(int64_t)g * Ktot + koff + (int64_t)k * n + i] : 0.0;
    u16 h, l;
    split_bf16(x, h, l);
    hi[dst_off + e] = h;
    lo[dst_off + e] = l;
  }
}
struct F_k_rsplit {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_rsplit_body(b, g, a...);
  }
};
__global__ void k_rsplit(const double* R, u16* hi, u16* lo, int N, int Np, int G, int64_t Ktot, int64_t koff,
                         int n, int64_t dst_off) {
  k_rsplit_body(blockIdx3(), gridDim3(), R, hi, lo, N, Np, G, Ktot, koff, n, dst_off);
}
void launch_rsplit(const DevState& s, hipStream_t st) {
  int64_t off = 0;
  for (int q = 0; q < s.nslots; ++q) {
    afq::glaunch<F_k_rsplit>(k_rsplit, dim3(2048), dim3(256), 0, st, s.R, s.Rb_hi, s.Rb_lo, s.N, s.Np, s.G, s.Ktot,
                       s.slot[q].koff, s.slot[q].n, off);
    off += (int64_t)s.G * s.slot[q].n * s.Np;
  }
}

// R_g hi parts in the fragment order of k_exchange_pw2 (see DevState::Rf): each
// (g, K step of 32, 16-row block) is 1 KB in lane order, so one wave's fragment load is
// one contiguous 1 KB read
__device__ __forceinline__ void k_rfrag_body(const uint3 bid_, const uint3 gdim_, const double* R, u16* out, u16* out_lo, int N, int G, int64_t Ktot, int64_t koff, int n, int nb,
                        int nks) {
  const int64_t total = (int64_t)G * nks * nb * 512;
  for (int64_t e = (int64_t)bid_.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gdim_.x * blockDim.x) {
    const int v = (int)(e & 7), lane = (int)((e >> 3) & 63);
    int64_t r = e >> 9;
    const int b = (int)(r % nb);
    r /= nb;
    const int ks = (int)(r % nks), g = (int)(r / nks);
    const int i = 16 * b + (lane & 15), k = 32 * ks + 8 * (lane >> 4) + v;
    const double x = (i < n && k < N) ? R[(int64_t)g * Ktot + koff + (int64_t)k * n + i] : 0.0;
    u16 h, l;
    split_bf16(x, h, l);
    out[e] = h;
    out_lo[e] = l;
  }
}
struct F_k_rfrag {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_rfrag_body(b, g, a...);
  }
};
__global__ void k_rfrag(const double* R, u16* out, u16* out_lo, int N, int G, int64_t Ktot, int64_t koff, int n, int nb,
                        int nks) {
  k_rfrag_body(blockIdx3(), gridDim3(), R, out, out_lo, N, G, Ktot, koff, n, nb, nks);
}
int64_t rfrag_elems(const DevState& s, int64_t* off) {
  const int Kp = (s.Np + 31) & ~31;
  if (Kp > PW2_KMAX) return 0;
  int64_t tot = 0;
  for (int q = 0; q < s.nslots; ++q) {
    if (s.slot[q].n > 64) return 0;
    if (off) off[q] = tot;
    tot += (int64_t)s.G * (Kp / 32) * ((s.slot[q].n + 15) / 16) * 512;
  }
  return tot;
}
void launch_rfrag(const DevState& s, hipStream_t st) {
  const int Kp = (s.Np + 31) & ~31;
  for (int q = 0; q < s.nslots; ++q)
    afq::glaunch<F_k_rfrag>(k_rfrag, dim3(2048), dim3(256), 0, st, s.R, s.Rf + s.rf_off[q], s.Rf_lo + s.rf_off[q], s.N, s.G,
                       s.Ktot, s.slot[q].koff,
                       s.slot[q].n, (s.slot[q].n + 15) / 16, Kp / 32);
}

// transpose + split theta of the selected walkers (one workgroup per walker and slot)
// into Tb[w][re/im][slot][j][k]: every (walker, component) row holds the slots'
// columns back to back, so the force bias reads it as one K-contiguous row and the
// exchange reads each (walker, component, slot, j) as a K-contiguous column
__device__ __forceinline__ void k_theta_split_body(const uint3 bid_, const uint3 gdim_, const double* theta, const int* sel, const int* nsel_dev,
                                                     u16* hi, u16* lo, int N,
                                                     int Np, int64_t Ktot, Slot s0, Slot s1, int ctot,
                                                     const int* skip) {
  __shared__ double tile[32 * 129];
  if (nsel_dev && (int)bid_.x >= *nsel_dev) return;
  const int w = sel ? sel[bid_.x] : bid_.x;
  if (skip && skip[w]) return;   // split already (by k_theta)
  const Slot sl = bid_.y == 0 ? s0 : s1;
  const int n2 = 2 * sl.n;
  const int coff = bid_.y == 0 ? 0 : 2 * s0.n;
  const double* th = theta + (int64_t)w * 2 * Ktot + 2 * sl.koff;
  for (int r0 = 0; r0 < Np; r0 += 32) {
    for (int e = threadIdx.x; e < 32 * n2; e += blockDim.x) {
      const int r = e / n2, c = e - r * n2;
      tile[r * 129 + c] = (r0 + r < N) ? th[(int64_t)(r0 + r) * n2 + c] : 0.0;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 32 * n2; e += blockDim.x) {
      const int c = e / 32, r = e - c * 32;
      if (r0 + r < Np) {
        u16 h, l;
        split_bf16(tile[r * 129 + c], h, l);
        const int64_t a = (((int64_t)w * 2 + (c & 1)) * (ctot / 2) + coff / 2 + (c >> 1)) * Np + r0 + r;
        hi[a] = h;
        lo[a] = l;
      }
    }
    __syncthreads();
  }
}
struct F_k_theta_split {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_theta_split_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_theta_split(const double* theta, const int* sel, const int* nsel_dev,
                                                     u16* hi, u16* lo, int N,
                                                     int Np, int64_t Ktot, Slot s0, Slot s1, int ctot,
                                                     const int* skip) {
  k_theta_split_body(blockIdx3(), gridDim3(), theta, sel, nsel_dev, hi, lo, N, Np, Ktot, s0, s1, ctot, skip);
}
void launch_theta_split(const DevState& s, const int* sel, int nsel, hipStream_t st, const int* nsel_dev) {
  afq::glaunch<F_k_theta_split>(k_theta_split, dim3(nsel, s.nslots), dim3(256), 0, st, s.theta, sel, nsel_dev, s.Tb_hi, s.Tb_lo, s.N,
                     s.Np, s.Ktot, s.slot[0], s.slot[s.nslots > 1 ? 1 : 0], s.ctot, (const int*)nullptr);
}

// Xp as k_exchange, f = R_g theta from bf16 hi/lo operands (NS = 2: BF16x3, NS = 1: BF16),
// FP32 accumulation, the f_ij f_ji reduction in FP64.
template <int NS>
__device__ __forceinline__ void k_exchange_bf16_body(const uint3 bid_, const uint3 gdim_, const u16* Rh, const u16* Rl, const u16* Th,
                                                                        const u16* Tl, const int* sel,
                                                          const int* nsel_dev, double* Xp, int Np, int GE, int nw, int W,
                                                          int G, Slot s0, Slot s1, int ctot, int ngt, int gridx,
                                                          int gridy, int gridz) {
  // one pass: 32-deep double-buffered stages (one barrier per stage) within 128 VGPRs
  // and 40 KB of LDS, four workgroups per CU
  using Eng = MmaBF16<XC_BM, XC_BN, 2, 2, NS, NS, (NS == 1 ? 32 : 64), NS == 1>;
  // f of the whole tile at once when it fits in the engine's LDS (NS = 2); else one
  // g-block at a time; the group sums' scratch follows f
  constexpr int LDF = XC_BN + 2;
  constexpr bool ONE_PASS = XC_BM * LDF * 4 + 64 <= Eng::LDS_BYTES;
  constexpr int FT_BYTES = (ONE_PASS ? XC_BM : XC_BM / 2) * LDF * 4;
  constexpr int LDSB = Eng::LDS_BYTES > FT_BYTES + 64 ? Eng::LDS_BYTES : FT_BYTES + 64;
  __shared__ __attribute__((aligned(16))) unsigned char lds[LDSB];
  double* red = reinterpret_cast<double*>(lds + FT_BYTES);
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, gridz, NS == 1 ? 32 : 8);   // walkers per L2 group
  const int zs = gridz > 1 ? tl.z : 0;
  const Slot sl = zs == 0 ? s0 : s1;
  const int n = sl.n, gt = XC_BM / n, wt = XC_BN / (2 * n);
  const int g0 = tl.x * gt, w0 = tl.y * wt;
  if (nsel_dev) nw = *nsel_dev;
  if (w0 >= nw) return;
  const int coff = (zs == 0 && sl.koff == s0.koff) ? 0 : 2 * s0.n;
  const int64_t roff = (zs == 0 && sl.koff == s0.koff) ? 0 : (int64_t)G * s0.n * Np;
  Eng e;
  e.run(
      [&](int c, int r) -> const u16* {
        const int gl = r / n, i = r - gl * n, g = g0 + gl;
        if (gl >= gt || g >= GE) return nullptr;
        return (c ? Rl : Rh) + roff + ((int64_t)g * n + i) * Np;
      },
      [&](int c, int q) -> const u16* {
        const int wl = q / (2 * n), cc = q - wl * 2 * n;
        if (wl >= wt || w0 + wl >= nw) return nullptr;
        const int w = sel ? sel[w0 + wl] : w0 + wl;
        return (c ? Tl : Th) + (((int64_t)w * 2 + (cc & 1)) * (ctot / 2) + coff / 2 + (cc >> 1)) * Np;
      },
      Np, lds);
  // g-blocks past GE hold zeros (their A rows are zero)
  float* F = reinterpret_cast<float*>(lds);
  const XPairsF<typename std::conditional<NS == 1, float, double>::type> xp(wt);
  double accr = 0.0, acci = 0.0;
  if (ONE_PASS) {
    const int rows = gt * n;
    e.store([&](int r, int c, float v) {
      if (r < rows) F[r * LDF + c] = v;
    });
    __syncthreads();
    xp.add(F, LDF, n, gt, wt, accr, acci);
  } else {
    for (int gl = 0; gl < gt; ++gl) {
      if (g0 + gl >= GE) break;
      e.store([&](int r, int c, float v) {
        const int rr = r - gl * n;
        if (rr >= 0 && rr < n) F[rr * LDF + c] = v;
      });
      __syncthreads();
      xp.add(F, LDF, n, 1, wt, accr, acci);
      __syncthreads();
    }
  }
  if (xp.finish(accr, acci, red) && xp.wl < wt && w0 + xp.wl < nw) {
    const int w = sel ? sel[w0 + xp.wl] : w0 + xp.wl;
    double* o = Xp + 2 * (((int64_t)zs * W + w) * ngt + tl.x);
    o[0] = accr;
    o[1] = acci;
  }
}
template <int NS>
struct F_k_exchange_bf16 {
  static constexpr int NT = 256, OCC = NS == 1 ? 4 : 2;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_exchange_bf16_body<NS>(b, g, a...);
  }
};
template <int NS>
__global__ __launch_bounds__(256, NS == 1 ? 4 : 2) void k_exchange_bf16(const u16* Rh, const u16* Rl, const u16* Th,
                                                                        const u16* Tl, const int* sel,
                                                          const int* nsel_dev, double* Xp, int Np, int GE, int nw, int W,
                                                          int G, Slot s0, Slot s1, int ctot, int ngt, int gridx,
                                                          int gridy, int gridz) {
  k_exchange_bf16_body<NS>(blockIdx3(), gridDim3(), Rh, Rl, Th, Tl, sel, nsel_dev, Xp, Np, GE, nw, W, G, s0, s1, ctot, ngt, gridx, gridy, gridz);
}

// One-pass BF16 exchange with the pair sums sum_ij f_ij f_ji in registers.  A workgroup
// takes one (live walker, slot) and a chunk of the Cholesky vectors: the walker's theta
// for the slot (both components, rows zero-padded to 16 NB, K to a multiple of 32)
// stays in LDS for the whole chunk, and each wave takes its own g's, reading R_g's rows
// straight into MFMA fragments.  For every pair of 16-row blocks I <= J of
// f_c = R_g theta_c^T (c = re, im) the wave forms X_c = f_c[I,J] (A = R_I,
// B = theta_c,J) and Y_c = f_c[J,I]^T (A = theta_c,I, B = R_J), which share a register
// layout, so the pair's sum_ab f[I,J]_ab f[J,I]_ba is an elementwise product of
// registers (off-diagonal pairs count twice, and the diagonal blocks are formed twice:
// 25% more MFMA at NB = 4) with no LDS round trip.  Padded rows of theta are zero, so
// the clamped (finite) R rows and K columns past the data contribute nothing.  The
// loads have no branches and run two K stages ahead.  Eight waves, two per
// SIMD: the two waves of a pair take the same g's and split the block pairs, so each
// holds half the accumulators.  The per-g-tile partials go to LDS and leave at the end
// in the layout of k_exchange_bf16's.
constexpr int PW_WAVES = 8, PW_STREAMS = 4, PW_KMAX = 512;
template <int NB>
__device__ __forceinline__ void k_exchange_pw_body(const uint3 bid_, const uint3 gdim_, const u16* __restrict__ Rh,
                                                                 const u16* __restrict__ Th, const int* sel,
                                                                 const int* nsel_dev, double* Xp, int Np, int GE,
                                                                 int nw, int W, int G,
                                                                 Slot s0, Slot s1, int ctot, int ngt_cap, int gt,
                                                                 int tpc, int nz, int nchunk) {
  constexpr int ROWS = 16 * NB;
  constexpr int NPAIR = NB * (NB + 1) / 2, NPH = (NPAIR + 1) / 2;   // block pairs, per wave of a pair
  __shared__ __attribute__((aligned(16))) u16 Ts[2 * ROWS * (PW_KMAX + 8)];
  __shared__ double part[2][PW_TMAX][2];
  const int Kp = (Np + 31) & ~31, nks = Kp >> 5, LDK = Kp + 8;
  const TileId tl = tile_id_at(bid_.x, nw * nz, 1, nchunk, 1);
  const int zs = tl.x % nz, l = tl.x / nz, chunk = tl.z;
  if (nsel_dev && l >= *nsel_dev) return;
  const Slot sl = zs == 0 ? s0 : s1;
  const int n = sl.n;
  const int coff = (zs == 0 && sl.koff == s0.koff) ? 0 : s0.n;
  const int64_t roff = (zs == 0 && sl.koff == s0.koff) ? 0 : (int64_t)G * s0.n * Np;
  const int w = sel ? sel[l] : l;
  const int ngt = (GE + gt - 1) / gt, t0 = chunk * tpc, t1 = min(ngt, t0 + tpc);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = wave & 1, u = wave >> 1;   // block-pair half, g stream
  const int cl = lane & 15, kh = lane >> 4;
  // theta of (w, slot) -> LDS [comp][row][LDK], zero outside the data
  for (int e = tid; e < 2 * ROWS * (LDK / 8); e += 64 * PW_WAVES) {
    const int k8 = e % (LDK / 8), rr = e / (LDK / 8), comp = rr / ROWS, j = rr - comp * ROWS;
    uint4 v = uint4{0u, 0u, 0u, 0u};
    if (j < n && 8 * k8 < Np)
      v = *reinterpret_cast<const uint4*>(Th + (((int64_t)w * 2 + comp) * (ctot / 2) + coff + j) * Np + 8 * k8);
    *reinterpret_cast<uint4*>(Ts + (comp * ROWS + j) * LDK + 8 * k8) = v;
  }
  for (int e = tid; e < 2 * PW_TMAX * 2; e += 64 * PW_WAVES) (&part[0][0][0])[e] = 0.0;
  __syncthreads();
  // this wave's g's: g-tiles t = t0 + u, t0 + u + PW_STREAMS, ..., gt g's each; both waves
  // of a stream take the same g's and split the block pairs (p even / odd)
  const int ntw = t1 - t0 > u ? (t1 - t0 - u + PW_STREAMS - 1) / PW_STREAMS : 0;
  const int ng = ntw * gt;
  auto g_of = [&](int gi) { return min((t0 + u + PW_STREAMS * (gi / gt)) * gt + gi % gt, GE - 1); };
  const u16* Rs = Rh + roff;
  int roffs[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) roffs[b] = min(16 * b + cl, n - 1) * Np;
  // R and theta fragments run two stages ahead in three register sets
  bf16x8 Ra[3][NB], Ta[3][2][NB];
  auto loadR = [&](int g, int ks, int set) {
    const u16* base = Rs + (int64_t)g * n * Np;   // wave-uniform
    const int kk = min(32 * ks + 8 * kh, Np - 8);
#pragma unroll
    for (int b = 0; b < NB; ++b) Ra[set][b] = *reinterpret_cast<const bf16x8*>(base + roffs[b] + kk);
  };
  auto loadT = [&](int ks, int set) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int b = 0; b < NB; ++b)
        Ta[set][c][b] = *reinterpret_cast<const bf16x8*>(Ts + (c * ROWS + 16 * b + cl) * LDK + 32 * ks + 8 * kh);
  };
  f32x4 X[NPH][2], Y[NPH][2];
  auto zero = [&]() {
#pragma unroll
    for (int h = 0; h < NPH; ++h)
#pragma unroll
      for (int c = 0; c < 2; ++c) X[h][c] = Y[h][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  // the block pairs (I <= J) in order p = 0 .. NPAIR-1; this wave takes p = 2 h + Q
  auto mma_half = [&](auto Qc, int rs, int ts) {
    constexpr int Q = decltype(Qc)::value;
    int p = 0;
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int J = I; J < NB; ++J, ++p)
        if ((p & 1) == Q)
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            X[p >> 1][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Ra[rs][I], Ta[ts][c][J], X[p >> 1][c], 0, 0, 0);
            Y[p >> 1][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Ta[ts][c][I], Ra[rs][J], Y[p >> 1][c], 0, 0, 0);
          }
  };
  auto pair_sum = [&](auto Qc, float& sr, float& si) {
    constexpr int Q = decltype(Qc)::value;
    int p = 0;
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int J = I; J < NB; ++J, ++p)
        if ((p & 1) == Q) {
          float ar = 0.f, ai = 0.f;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            ar += X[p >> 1][0][r] * Y[p >> 1][0][r] - X[p >> 1][1][r] * Y[p >> 1][1][r];
            ai += X[p >> 1][0][r] * Y[p >> 1][1][r] + X[p >> 1][1][r] * Y[p >> 1][0][r];
          }
          const float m = I == J ? 1.f : 2.f;
          sr += m * ar;
          si += m * ai;
        }
  };
  // the whole stage loop for one half of the block pairs (one copy per half, so that
  // neither loop branches on the half)
  auto run = [&](auto Qc) {
    double pr = 0.0, pi = 0.0;   // this lane's share of the current g-tile
    auto finish_g = [&](int gi) {
      if (gi >= ng) return;   // a padding stage
      float sr = 0.f, si = 0.f;
      pair_sum(Qc, sr, si);
      const int tw = gi / gt, g = (t0 + u + PW_STREAMS * tw) * gt + gi % gt;
      if (g < GE) {
        pr += (double)sr;
        pi += (double)si;
      }
      if (gi % gt == gt - 1) {   // last g of the tile
        const double a = wave_sum(pr), b = wave_sum(pi);
        if (lane == 0) {
          part[q][u + PW_STREAMS * tw][0] = a;
          part[q][u + PW_STREAMS * tw][1] = b;
        }
        pr = pi = 0.0;
      }
      zero();
    };
    // stages (gi, ks) in order, stage s in register set s % 3; the count is rounded up to
    // a multiple of 3 with padding stages (their loads re-read the last g, their products
    // are never used), so the loop has no branch around loads
    const int nst = ng * nks;
    zero();
    int gR = 0, kR = 0;   // the stage whose fragments are requested next
    auto advance = [&](int& g, int& k) {
      if (++k == nks) { k = 0; ++g; }
    };
    if (nst > 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        loadR(g_of(min(gR, ng - 1)), kR, i);
        loadT(kR, i);
        advance(gR, kR);
      }
    }
    int gi = 0, ks = 0;
    for (int s = 0; s < nst; s += 3) {
#pragma unroll
      for (int h = 0; h < 3; ++h) {
        loadR(g_of(min(gR, ng - 1)), kR, (h + 2) % 3);
        loadT(kR, (h + 2) % 3);
        advance(gR, kR);
        mma_half(Qc, h, h);
        if (ks == nks - 1) finish_g(gi);
        advance(gi, ks);
      }
    }
  };
  if (q == 0) run(std::integral_constant<int, 0>{});
  else run(std::integral_constant<int, 1>{});
  __syncthreads();
  double* o = Xp + 2 * (((int64_t)zs * W + w) * ngt_cap);
  for (int t = t0 + tid; t < t1; t += 64 * PW_WAVES) {
    o[2 * t] = part[0][t - t0][0] + part[1][t - t0][0];
    o[2 * t + 1] = part[0][t - t0][1] + part[1][t - t0][1];
  }
}
template <int NB>
struct F_k_exchange_pw {
  static constexpr int NT = 64 * PW_WAVES, OCC = 1;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_exchange_pw_body<NB>(b, g, a...);
  }
};
template <int NB>
__global__ __launch_bounds__(64 * PW_WAVES, 1) void k_exchange_pw(const u16* __restrict__ Rh,
                                                                 const u16* __restrict__ Th, const int* sel,
                                                                 const int* nsel_dev, double* Xp, int Np, int GE,
                                                                 int nw, int W, int G,
                                                                 Slot s0, Slot s1, int ctot, int ngt_cap, int gt,
                                                                 int tpc, int nz, int nchunk) {
  k_exchange_pw_body<NB>(blockIdx3(), gridDim3(), Rh, Th, sel, nsel_dev, Xp, Np, GE, nw, W, G, s0, s1, ctot, ngt_cap, gt, tpc, nz, nchunk);
}

static void launch_exchange_q8(const DevState& s, const int* sel, int nsel, const int* nsel_dev, hipStream_t st);
// k_exchange_pw for the one-pass surrogate where it applies (slots of at most 64
// electrons, N padded to 32 at most PW_KMAX); false: use k_exchange_bf16
// x3: the three-pass split form of k_exchange_pw2 (false where it does not apply)
static bool exchange_pw(const DevState& s, const int* sel, int nsel, const int* nsel_dev, hipStream_t st,
                        bool x3 = false) {
  const int Kp = (s.Np + 31) & ~31;
  int nmax = 0;
  for (int z = 0; z < s.nslots; ++z) nmax = std::max(nmax, s.slot[z].n);
  if (Kp > PW_KMAX || nmax > 64 || nsel <= 0) return false;
  const bool v2 = s.Rf != nullptr && (x3 || s.xc_variant != 2);   // Rf is built where k_exchange_pw2 applies
  if (x3 && !v2) return false;
  auto go = [&](int z0, int nz, const u16* rh, const u16* th, double* xp, Slot a, Slot b) {
    const int nb = (a.n + 15) / 16;
    const int gt = exchange_tile_g(a.n), ngt = (int)cdivu(s.GE, gt);
    // chunks per (walker, spin): for k_exchange_pw2 one per 8 MB of the spin's R, at most 6
    // (its workgroups run spin-major, so the resident ones of an XCD share a chunk of one
    // spin's R; 6 measured fastest of 2 .. 20 at N=300, where R is 49 MB a spin; a smaller R
    // stays in L2 whole, and every further chunk only reloads the walker's theta), 4 for
    // k_exchange_pw.  Each g-tile's partial is stored on its own, so the chunking does not
    // change the result.
    const int64_t rbytes = (int64_t)s.GE * (16 * nb) * Kp * 2;
    const int want = s.xc_chunks > 0 ? s.xc_chunks
                                     : v2 ? (int)std::min<int64_t>(6, std::max<int64_t>(1, cdivu(rbytes, 8 << 20)))
                                          : 4;
    const int tpc = std::min(PW_TMAX, (int)cdivu(ngt, want)), nchunk = (int)cdivu(ngt, tpc);
    const dim3 grid((unsigned)(nsel * nz * nchunk));
    if (v2) {
      const u16* rf = s.Rf + s.rf_off[z0];
      const int64_t rfs = nz > 1 ? s.rf_off[1] - s.rf_off[0] : 0;
      const u16* rfl = s.Rf_lo + s.rf_off[z0];
      const u16* tl = s.Tb_lo + (th - s.Tb_hi);
      if (x3 && s.xc3_variant != 2)
        launch_exchange_pw2x3(rf, rfl, rfs, th, tl, sel, nsel_dev, xp, s.Np, s.GE, nsel, s.W, a, b, s.ctot, s.ngt_cap,
                              gt, tpc, nz, nchunk, nb, st);
      else
        launch_exchange_pw2(rf, rfl, rfs, th, tl, sel, nsel_dev, xp, s.Np, s.GE, nsel, s.W, a, b, s.ctot, s.ngt_cap,
                            gt, tpc, nz, nchunk, nb, s.xc_variant == 3 || x3 ? 4 : 8, x3, st);
      return;
    }
#define AFQ_PW(NB_)                                                                                            \
  afq::glaunch<F_k_exchange_pw<NB_>>(k_exchange_pw<NB_>, grid, dim3(64 * PW_WAVES), 0, st, rh, th, sel, nsel_dev, xp, s.Np, s.GE, nsel, \
                     s.W, s.G, a, b, s.ctot, s.ngt_cap, gt, tpc, nz, nchunk)
    switch (nb) {
      case 1: AFQ_PW(1); break;
      case 2: AFQ_PW(2); break;
      case 3: AFQ_PW(3); break;
      default: AFQ_PW(4); break;
    }
#undef AFQ_PW
  };
  if (s.nslots == 1 || s.slot[1].n == s.slot[0].n) {
    go(0, s.nslots, s.Rb_hi, s.Tb_hi, s.Xp, s.slot[0], s.nslots > 1 ? s.slot[1] : s.slot[0]);
  } else {
    go(0, 1, s.Rb_hi, s.Tb_hi, s.Xp, s.slot[0], s.slot[0]);
    Slot bb = s.slot[1];
    bb.koff = s.slot[0].koff;   // koff sentinel: offsets zero, pointers advanced instead
    go(1, 1, s.Rb_hi + (int64_t)s.G * s.slot[0].n * s.Np, s.Tb_hi + (int64_t)s.slot[0].n * s.Np,
       s.Xp + 2 * (int64_t)s.W * s.ngt_cap, bb, bb);
  }
  return true;
}

void launch_exchange_lp(const DevState& s, const int* sel, int nsel, int prec, hipStream_t st, const int* nsel_dev) {
  if (prec == AFQ_PREC_FP8) {
    launch_exchange_q8(s, sel, nsel, nsel_dev, st);
    return;
  }
  if (!s.tb_live) launch_theta_split(s, sel, nsel, st, nsel_dev);   // else split by the force bias already
  if (prec == AFQ_PREC_BF16 && s.xc_variant != 1 && exchange_pw(s, sel, nsel, nsel_dev, st)) return;
  // the three-pass pair-wise kernel from 13 electrons a slot up: below, its 16-row blocks
  // are mostly padding and the tiled kernel is faster (256 walkers: 0.018 against 0.027 ms
  // at n = 4, even at n = 12, 0.36 against 0.62 ms at n = 24)
  int nmax3 = 0;
  for (int z = 0; z < s.nslots; ++z) nmax3 = std::max(nmax3, s.slot[z].n);
  if (prec == AFQ_PREC_BF16X3 && s.xc3_variant != 1 && nmax3 > 12 && exchange_pw(s, sel, nsel, nsel_dev, st, true))
    return;
  auto go = [&](int z0, int nz, double* xp) {
    const Slot& a = s.slot[z0];
    const int gt = exchange_tile_g(a.n), wt = exchange_tile_w(a.n);
    const int ngt = (int)cdivu(s.GE, gt), gy = (int)cdivu(nsel, wt);
    const Slot s1 = nz > 1 ? s.slot[1] : a;
    if (prec == AFQ_PREC_BF16X3)
      afq::glaunch<F_k_exchange_bf16<2>>(k_exchange_bf16<2>, dim3(ngt * gy * nz), dim3(256), 0, st, s.Rb_hi, s.Rb_lo, s.Tb_hi,
                         s.Tb_lo, sel, nsel_dev, xp, s.Np, s.GE, nsel, s.W, s.G, a, s1, s.ctot, s.ngt_cap, ngt, gy, nz);
    else
      afq::glaunch<F_k_exchange_bf16<1>>(k_exchange_bf16<1>, dim3(ngt * gy * nz), dim3(256), 0, st, s.Rb_hi, s.Rb_lo, s.Tb_hi,
                         s.Tb_lo, sel, nsel_dev, xp, s.Np, s.GE, nsel, s.W, s.G, a, s1, s.ctot, s.ngt_cap, ngt, gy, nz);
  };
  if (s.nslots == 1 || s.slot[1].n == s.slot[0].n) go(0, s.nslots, s.Xp);
  else {
    go(0, 1, s.Xp);
    // the second slot alone: present it as s0 with its own offsets
    const Slot& b = s.slot[1];
    const int gt = exchange_tile_g(b.n), wt = exchange_tile_w(b.n);
    const int ngt = (int)cdivu(s.GE, gt), gy = (int)cdivu(nsel, wt);
    // pass pointers advanced to slot 1's R rows / theta columns; koff sentinel makes coff/roff zero
    Slot bb = b;
    bb.koff = s.slot[0].koff;
    const u16* rh = s.Rb_hi + (int64_t)s.G * s.slot[0].n * s.Np;
    const u16* rl = s.Rb_lo + (int64_t)s.G * s.slot[0].n * s.Np;
    const u16* th = s.Tb_hi + (int64_t)s.slot[0].n * s.Np;
    const u16* tlo = s.Tb_lo + (int64_t)s.slot[0].n * s.Np;
    double* xp = s.Xp + 2 * (int64_t)s.W * s.ngt_cap;
    if (prec == AFQ_PREC_BF16X3)
      afq::glaunch<F_k_exchange_bf16<2>>(k_exchange_bf16<2>, dim3(ngt * gy), dim3(256), 0, st, rh, rl, th, tlo, sel, nsel_dev, xp, s.Np, s.GE,
                         nsel, s.W, s.G, bb, bb, s.ctot, s.ngt_cap, ngt, gy, 1);
    else
      afq::glaunch<F_k_exchange_bf16<1>>(k_exchange_bf16<1>, dim3(ngt * gy), dim3(256), 0, st, rh, rl, th, tlo, sel, nsel_dev, xp, s.Np, s.GE,
                         nsel, s.W, s.G, bb, bb, s.ctot, s.ngt_cap, ngt, gy, 1);
  }
}

// ------------------------------------------------------------------ FP8 (e4m3) exchange
// Operands in OCP e4m3 (1-4-3, bias 7, largest finite 448), each Cholesky vector g
// scaled by a power of two s_g (its largest |R_g| entry, over both slots, maps into
// (224, 448]) and each walker's theta of a slot by a power of two t; the products
// accumulate in FP32 on v_mfma_scale_f32_16x16x128_f8f6f4 (unit block scales) and
// the epilogue multiplies f by 1/(s_g t), exactly, before the pair sums.

// float -> e4m3, round to nearest even, saturating at 448
__device__ __forceinline__ unsigned f2e4m3(float x) {
  const unsigned sgn = (__float_as_uint(x) >> 24) & 0x80u;
  const float a = fabsf(x);
  if (!(a < 464.f)) return sgn | 0x7eu;
  if (a < 0.015625f) return sgn | (unsigned)rintf(a * 512.f);   // subnormals: multiples of 2^-9 (8 = 2^-6)
  const unsigned u = __float_as_uint(a);
  int e = (int)(u >> 23) - 127;
  const unsigned m = u & 0x7fffffu, rem = m & 0xfffffu;
  unsigned r = m >> 20;
  if (rem > 0x80000u || (rem == 0x80000u && (r & 1u))) ++r;
  if (r == 8u) { r = 0u; ++e; }
  if (e > 8 || (e == 8 && r == 7u)) { e = 8; r = 6u; }
  return sgn | ((unsigned)(e + 7) << 3) | r;
}
// the power of two s with amax * s in (224, 448] (1 for amax = 0)
__device__ __forceinline__ float e4m3_scale(float amax) {
  if (!(amax > 1e-30f)) return 1.f;
  int e;
  frexpf(448.f / amax, &e);   // 448/amax = f 2^e, f in [0.5, 1)
  return ldexpf(1.f, e - 1);
}
__device__ __forceinline__ float block_max(float v, float* red) {
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float m = 0.f;
  for (int q = 0; q < (int)(blockDim.x >> 6); ++q) m = fmaxf(m, red[q]);
  __syncthreads();
  return m;
}

// Rq[slot][g][i][Npq] = e4m3(s_g R_s,g(i, k)), rinv[g] = 1 / s_g; one workgroup per g
__device__ __forceinline__ void k_rq8_body(const uint3 bid_, const uint3 gdim_, const double* R, unsigned char* Rq, float* rinv, int N, int Npq, int G,
                                             int64_t Ktot, Slot s0, Slot s1, int nslots) {
  __shared__ float red[4];
  const int g = bid_.x;
  const double* Rg = R + (int64_t)g * Ktot;
  float amax = 0.f;
  for (int q = 0; q < nslots; ++q) {
    const Slot sl = q ? s1 : s0;
    for (int e = threadIdx.x; e < sl.n * N; e += blockDim.x) amax = fmaxf(amax, (float)fabs(Rg[sl.koff + e]));
  }
  const float sc = e4m3_scale(block_max(amax, red));
  if (threadIdx.x == 0) rinv[g] = 1.f / sc;
  int64_t off = 0;
  for (int q = 0; q < nslots; ++q) {
    const Slot sl = q ? s1 : s0;
    unsigned char* dst = Rq + off + (int64_t)g * sl.n * Npq;
    for (int e = threadIdx.x; e < sl.n * Npq; e += blockDim.x) {
      const int i = e / Npq, k = e - i * Npq;
      dst[e] = k < N ? (unsigned char)f2e4m3((float)(Rg[sl.koff + (int64_t)k * sl.n + i] * (double)sc)) : 0;
    }
    off += (int64_t)G * sl.n * Npq;
  }
}
struct F_k_rq8 {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_rq8_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_rq8(const double* R, unsigned char* Rq, float* rinv, int N, int Npq, int G,
                                             int64_t Ktot, Slot s0, Slot s1, int nslots) {
  k_rq8_body(blockIdx3(), gridDim3(), R, Rq, rinv, N, Npq, G, Ktot, s0, s1, nslots);
}

// Tq[w][re/im][slot][j][Npq] = e4m3(t theta_s[w][k][j]), tinv[w][slot] = 1 / t; one
// workgroup per (selected walker, slot)
__device__ __forceinline__ void k_theta_q8_body(const uint3 bid_, const uint3 gdim_, const double* theta, const int* sel, const int* nsel_dev,
                                                  unsigned char* Tq, float* tinv, int N, int Npq, int64_t Ktot, Slot s0,
                                                  Slot s1, int ctot) {
  __shared__ float red[4];
  if (nsel_dev && (int)bid_.x >= *nsel_dev) return;
  const int w = sel ? sel[bid_.x] : bid_.x;
  const Slot sl = bid_.y == 0 ? s0 : s1;
  const int n2 = 2 * sl.n;
  const int coff = bid_.y == 0 ? 0 : 2 * s0.n;
  const double* th = theta + (int64_t)w * 2 * Ktot + 2 * sl.koff;
  float amax = 0.f;
  for (int e = threadIdx.x; e < N * n2; e += blockDim.x) amax = fmaxf(amax, (float)fabs(th[e]));
  const float sc = e4m3_scale(block_max(amax, red));
  if (threadIdx.x == 0) tinv[2 * (int64_t)w + bid_.y] = 1.f / sc;
  for (int e = threadIdx.x; e < n2 * Npq; e += blockDim.x) {
    const int c = e / Npq, k = e - c * Npq;
    const int64_t a = (((int64_t)w * 2 + (c & 1)) * (ctot / 2) + coff / 2 + (c >> 1)) * Npq + k;
    Tq[a] = k < N ? (unsigned char)f2e4m3((float)(th[(int64_t)k * n2 + c] * (double)sc)) : 0;
  }
}
struct F_k_theta_q8 {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_theta_q8_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_theta_q8(const double* theta, const int* sel, const int* nsel_dev,
                                                  unsigned char* Tq, float* tinv, int N, int Npq, int64_t Ktot, Slot s0,
                                                  Slot s1, int ctot) {
  k_theta_q8_body(blockIdx3(), gridDim3(), theta, sel, nsel_dev, Tq, tinv, N, Npq, Ktot, s0, s1, ctot);
}

// Xp as k_exchange from the e4m3 operands: 128 x 128 tiles, four waves of 64 x 64, K
// stages of 128 (one v_mfma_scale_f32_16x16x128_f8f6f4 deep), register-prefetched.
// Lane l supplies 32 consecutive K bytes at 32 (l / 16) of row l % 16 for both A and
// B, so every product pairs equal k whatever the instruction's internal K order.
typedef int i32x8 __attribute__((ext_vector_type(8)));
constexpr int Q8_BK = 128, Q8_LDK = Q8_BK + 16;
__device__ __forceinline__ void k_exchange_q8_body(const uint3 bid_, const uint3 gdim_, const unsigned char* Rq, const unsigned char* Tq,
                                                        const float* rinv, const float* tinv, const int* sel,
                                                        const int* nsel_dev, double* Xp, int Npq, int GE, int nw, int W,
                                                        int G, Slot s0,
                                                        Slot s1, int ctot, int ngt_cap, int gridx, int gridy,
                                                        int gridz) {
  constexpr int LDF = XC_BN + 2;
  constexpr int STAGE = 2 * XC_BM * Q8_LDK, FT = (XC_BM / 2) * LDF * 4;
  __shared__ __attribute__((aligned(16))) unsigned char lds[STAGE > FT ? STAGE : FT];
  __shared__ double red[8];
  unsigned char* As = lds;
  unsigned char* Bs = lds + XC_BM * Q8_LDK;
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, gridz, 8);
  const int zs = gridz > 1 ? tl.z : 0;
  const Slot sl = zs == 0 ? s0 : s1;
  const int n = sl.n, gt = XC_BM / n, wt = XC_BN / (2 * n);
  const int g0 = tl.x * gt, w0 = tl.y * wt;
  if (nsel_dev) nw = *nsel_dev;
  if (w0 >= nw) return;
  const int coff = (zs == 0 && sl.koff == s0.koff) ? 0 : 2 * s0.n;
  const int64_t roff = (zs == 0 && sl.koff == s0.koff) ? 0 : (int64_t)G * s0.n * Npq;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 1, wn = wave & 1;
  // 16-byte chunks: thread -> rows (tid >> 3) + 32 q, chunk (tid & 7) of the 128-byte stage
  const int ch = tid & 7;
  const unsigned char* pA[4];
  const unsigned char* pB[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = (tid >> 3) + 32 * q;
    const int gl = r / n, i = r - gl * n, g = g0 + gl;
    pA[q] = (gl < gt && g < GE) ? Rq + roff + ((int64_t)g * n + i) * Npq + 16 * ch : nullptr;
    const int wl = r / (2 * n), cc = r - wl * 2 * n;
    pB[q] = nullptr;
    if (wl < wt && w0 + wl < nw) {
      const int w = sel ? sel[w0 + wl] : w0 + wl;
      pB[q] = Tq + (((int64_t)w * 2 + (cc & 1)) * (ctot / 2) + coff / 2 + (cc >> 1)) * Npq + 16 * ch;
    }
  }
  uint4 ra[4], rb[4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ra[q] = uint4{0u, 0u, 0u, 0u};
      rb[q] = uint4{0u, 0u, 0u, 0u};
      if (k0 + 16 * ch < Npq) {
        if (pA[q]) ra[q] = *reinterpret_cast<const uint4*>(pA[q] + k0);
        if (pB[q]) rb[q] = *reinterpret_cast<const uint4*>(pB[q] + k0);
      }
    }
  };
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nst = (Npq + Q8_BK - 1) / Q8_BK;
  fetch(0);
  for (int st = 0; st < nst; ++st) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = (tid >> 3) + 32 * q;
      *reinterpret_cast<uint4*>(As + r * Q8_LDK + 16 * ch) = ra[q];
      *reinterpret_cast<uint4*>(Bs + r * Q8_LDK + 16 * ch) = rb[q];
    }
    __syncthreads();
    if (st + 1 < nst) fetch((st + 1) * Q8_BK);
    const int koff = 32 * (lane >> 4);
    i32x8 a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned char* pa = As + (wm * 64 + i * 16 + (lane & 15)) * Q8_LDK + koff;
      const uint4 lo = *reinterpret_cast<const uint4*>(pa), hi = *reinterpret_cast<const uint4*>(pa + 16);
      a[i] = i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
      const unsigned char* pb = Bs + (wn * 64 + i * 16 + (lane & 15)) * Q8_LDK + koff;
      const uint4 lb = *reinterpret_cast<const uint4*>(pb), hb = *reinterpret_cast<const uint4*>(pb + 16);
      b[i] = i32x8{(int)lb.x, (int)lb.y, (int)lb.z, (int)lb.w, (int)hb.x, (int)hb.y, (int)hb.z, (int)hb.w};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a[i], b[j], acc[i][j], 0, 0, 0, 127, 0, 127);
    __syncthreads();
  }
  // unscale while storing f: row -> Cholesky vector g0 + gl, column -> walker w0 + c / 2n
  float* F = reinterpret_cast<float*>(lds);
  float cs[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = wn * 64 + j * 16 + (lane & 15), wl = c / (2 * n);
    cs[j] = 0.f;
    if (wl < wt && w0 + wl < nw) {
      const int w = sel ? sel[w0 + wl] : w0 + wl;
      cs[j] = tinv[2 * (int64_t)w + zs];
    }
  }
  const XPairsF<float> xp(wt);
  double accr = 0.0, acci = 0.0;
  for (int gl = 0; gl < gt; ++gl) {
    if (g0 + gl >= GE) break;
    const float rs = rinv[g0 + gl];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int rr = wm * 64 + i * 16 + 4 * (lane >> 4) + r - gl * n;
          if (rr >= 0 && rr < n) F[rr * LDF + wn * 64 + j * 16 + (lane & 15)] = acc[i][j][r] * rs * cs[j];
        }
    __syncthreads();
    xp.add(F, LDF, n, 1, wt, accr, acci);
    __syncthreads();
  }
  if (xp.finish(accr, acci, red) && xp.wl < wt && w0 + xp.wl < nw) {
    const int w = sel ? sel[w0 + xp.wl] : w0 + xp.wl;
    double* o = Xp + 2 * (((int64_t)zs * W + w) * ngt_cap + tl.x);
    o[0] = accr;
    o[1] = acci;
  }
}
struct F_k_exchange_q8 {
  static constexpr int NT = 256, OCC = 2;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_exchange_q8_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256, 2) void k_exchange_q8(const unsigned char* Rq, const unsigned char* Tq,
                                                        const float* rinv, const float* tinv, const int* sel,
                                                        const int* nsel_dev, double* Xp, int Npq, int GE, int nw, int W,
                                                        int G, Slot s0,
                                                        Slot s1, int ctot, int ngt_cap, int gridx, int gridy,
                                                        int gridz) {
  k_exchange_q8_body(blockIdx3(), gridDim3(), Rq, Tq, rinv, tinv, sel, nsel_dev, Xp, Npq, GE, nw, W, G, s0, s1, ctot, ngt_cap, gridx, gridy, gridz);
}

void launch_rq8(const DevState& s, hipStream_t st) {
  afq::glaunch<F_k_rq8>(k_rq8, dim3(s.G), dim3(256), 0, st, s.R, s.Rq8, s.rinv8, s.N, s.Npq, s.G, s.Ktot, s.slot[0],
                     s.slot[s.nslots > 1 ? 1 : 0], s.nslots);
}

static void launch_exchange_q8(const DevState& s, const int* sel, int nsel, const int* nsel_dev, hipStream_t st) {
  afq::glaunch<F_k_theta_q8>(k_theta_q8, dim3(nsel, s.nslots), dim3(256), 0, st, s.theta, sel, nsel_dev, s.Tq8, s.tinv8, s.N, s.Npq,
                     s.Ktot, s.slot[0], s.slot[s.nslots > 1 ? 1 : 0], s.ctot);
  auto go = [&](const unsigned char* rq, const unsigned char* tq, const float* ti, double* xp, Slot a, Slot b, int nz) {
    const int gt = exchange_tile_g(a.n), wt = exchange_tile_w(a.n);
    const int ngt = (int)cdivu(s.GE, gt), gy = (int)cdivu(nsel, wt);
    afq::glaunch<F_k_exchange_q8>(k_exchange_q8, dim3(ngt * gy * nz), dim3(256), 0, st, rq, tq, s.rinv8, ti, sel, nsel_dev, xp, s.Npq,
                       s.GE, nsel, s.W, s.G, a, b, s.ctot, s.ngt_cap, ngt, gy, nz);
  };
  if (s.nslots == 1 || s.slot[1].n == s.slot[0].n) {
    go(s.Rq8, s.Tq8, s.tinv8, s.Xp, s.slot[0], s.nslots > 1 ? s.slot[1] : s.slot[0], s.nslots);
  } else {
    go(s.Rq8, s.Tq8, s.tinv8, s.Xp, s.slot[0], s.slot[0], 1);
    // the second slot alone, presented as s0 with pointers advanced to its rows and columns;
    // its theta scales sit at tinv[2w + 1]
    Slot bb = s.slot[1];
    bb.koff = s.slot[0].koff;
    go(s.Rq8 + (int64_t)s.G * s.slot[0].n * s.Npq, s.Tq8 + (int64_t)s.slot[0].n * s.Npq, s.tinv8 + 1,
       s.Xp + 2 * (int64_t)s.W * s.ngt_cap, bb, bb, 1);
  }
}

// ------------------------------------------------------------------ mixed-precision force bias
// fb[w][g][c] = alpha sum_{s,i,k} Tb[w][c][s][i][k] Rb[s][g][i][k]: rows (w, c) of the
// split theta against rows g of the split rotated Cholesky, one K-contiguous run of
// n_s * Np per slot, FP32 accumulation.  With part, each workgroup takes one slot
// (grid z = slot) and stores its FP32 sum to part[slot][row][g]; k_fb_combine adds the
// two in FP64.  The split doubles the workgroups: 640 tiles at 4096 walkers and G = 1200
// fill 1.25 rounds of the 512 resident slots, 1280 fill 2.5.
template <int NS>
__device__ __forceinline__ void k_force_bias_bf16_body(const uint3 bid_, const uint3 gdim_, const u16* Rh, const u16* Rl, const u16* Th,
                                                            const u16* Tl, double* fb, const int* live,
                                                            const int* nlive, int G, int Np, int nsum, int nslots,
                                                            Slot s0, Slot s1, double alpha, int gridx, int gridy,
                                                            float* part, int prow) {
  using Eng = MmaBF16<128, 128, 2, 2, NS, NS, 32, false, true>;
  __shared__ __attribute__((aligned(16))) unsigned char lds[Eng::LDS_BYTES];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, part ? nslots : 1, 8);
  const int row0 = tl.y * 128, g0 = tl.x * 128;
  const int nrow = 2 * *nlive;   // live walkers only, as the FP64 force bias
  if (row0 >= nrow) return;
  Eng e;
  int64_t roff = 0;
  int coff = 0;
  const int zlo = part ? tl.z : 0, zhi = part ? tl.z + 1 : nslots;
  for (int z = 0; z < zlo; ++z) {
    const int n = z == 0 ? s0.n : s1.n;
    roff += (int64_t)G * n * Np;
    coff += n;
  }
  for (int z = zlo; z < zhi; ++z) {
    const int n = z == 0 ? s0.n : s1.n;
    const int64_t ro = roff;
    const int co = coff;
    e.run(
        [&](int c, int r) -> const u16* {
          const int q = row0 + r;
          if (q >= nrow) return nullptr;
          return (c ? Tl : Th) + ((int64_t)(2 * live[q >> 1] + (q & 1)) * nsum + co) * Np;
        },
        [&](int c, int col) -> const u16* {
          const int g = g0 + col;
          if (g >= G) return nullptr;
          return (c ? Rl : Rh) + ro + (int64_t)g * n * Np;
        },
        n * Np, lds);
    __syncthreads();
    roff += (int64_t)G * n * Np;
    coff += n;
  }
  if (part) {
    float* o = part + (int64_t)zlo * prow * G;
    e.store([&](int r, int c, float v) {
      const int q = row0 + r, g = g0 + c;
      if (q < nrow && g < G) o[(int64_t)q * G + g] = v;
    });
    return;
  }
  e.store([&](int r, int c, float v) {
    const int q = row0 + r, g = g0 + c;
    if (q < nrow && g < G) fb[(int64_t)live[q >> 1] * 2 * G + 2 * g + (q & 1)] = alpha * (double)v;
  });
}
template <int NS>
struct F_k_force_bias_bf16 {
  static constexpr int NT = 256, OCC = 2;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_force_bias_bf16_body<NS>(b, g, a...);
  }
};
template <int NS>
__global__ __launch_bounds__(256, 2) void k_force_bias_bf16(const u16* Rh, const u16* Rl, const u16* Th,
                                                            const u16* Tl, double* fb, const int* live,
                                                            const int* nlive, int G, int Np, int nsum, int nslots,
                                                            Slot s0, Slot s1, double alpha, int gridx, int gridy,
                                                            float* part, int prow) {
  k_force_bias_bf16_body<NS>(blockIdx3(), gridDim3(), Rh, Rl, Th, Tl, fb, live, nlive, G, Np, nsum, nslots, s0, s1, alpha, gridx, gridy, part, prow);
}

// fb of the live walkers from the two slots' FP32 partial sums (added in FP64)
__device__ __forceinline__ void k_fb_combine_body(const uint3 bid_, const uint3 gdim_, const float* __restrict__ part,
                                                  double* __restrict__ fb, const int* live, const int* nlive, int G,
                                                  int prow, double alpha) {
  const int64_t i = (int64_t)bid_.x * blockDim.x + threadIdx.x;
  const int nrow = 2 * *nlive;
  if (i >= (int64_t)nrow * G) return;
  const int q = (int)(i / G), g = (int)(i - (int64_t)q * G);
  const double v = (double)part[i] + (double)part[(int64_t)prow * G + i];
  fb[(int64_t)live[q >> 1] * 2 * G + 2 * g + (q & 1)] = alpha * v;
}
struct F_k_fb_combine {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_fb_combine_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_fb_combine(const float* __restrict__ part, double* __restrict__ fb,
                                                    const int* live, const int* nlive, int G, int prow, double alpha) {
  k_fb_combine_body(blockIdx3(), gridDim3(), part, fb, live, nlive, G, prow, alpha);
}

void launch_force_bias_lp(const DevState& s, int prec, hipStream_t st) {
  launch_live_list(s, st);
  // the live walkers k_theta split straight after their theta are skipped
  afq::glaunch<F_k_theta_split>(k_theta_split, dim3(s.W, s.nslots), dim3(256), 0, st, s.theta, s.live, s.nlive, s.Tb_hi,
                     s.Tb_lo, s.N, s.Np, s.Ktot, s.slot[0], s.slot[s.nslots > 1 ? 1 : 0], s.ctot,
                     (const int*)(s.tb_post ? s.gfresh : nullptr));
  s.tb_post = false;
  s.tb_live = true;
  const int gx = (int)cdivu(s.G, 128), gy = (int)cdivu(2 * (int64_t)s.W, 128);
  const Slot& b = s.slot[s.nslots > 1 ? 1 : 0];
  // the two-slot split needs the partial buffer sized for this population
  float* part = s.nslots == 2 && s.fbp && s.fbp_rows >= 2 * s.W && s.fb_split ? s.fbp : nullptr;
  const int nz = part ? 2 : 1;
  if (prec == AFQ_PREC_BF16X3)
    afq::glaunch<F_k_force_bias_bf16<2>>(k_force_bias_bf16<2>, dim3(gx * gy * nz), dim3(256), 0, st, s.Rb_hi, s.Rb_lo,
                                         s.Tb_hi, s.Tb_lo, s.fb, s.live, s.nlive, s.G, s.Np, s.ctot / 2, s.nslots,
                                         s.slot[0], b, (double)s.slot[0].mult, gx, gy, part, s.fbp_rows);
  else
    afq::glaunch<F_k_force_bias_bf16<1>>(k_force_bias_bf16<1>, dim3(gx * gy * nz), dim3(256), 0, st, s.Rb_hi, s.Rb_lo,
                                         s.Tb_hi, s.Tb_lo, s.fb, s.live, s.nlive, s.G, s.Np, s.ctot / 2, s.nslots,
                                         s.slot[0], b, (double)s.slot[0].mult, gx, gy, part, s.fbp_rows);
  if (part)
    afq::glaunch<F_k_fb_combine>(k_fb_combine, dim3(cdivu(2 * (int64_t)s.W * s.G, 256)), dim3(256), 0, st, part, s.fb,
                                 s.live, s.nlive, s.G, s.fbp_rows, (double)s.slot[0].mult);
}

// ------------------------------------------------------------------ mixed-precision VHS
// Lt[t][g] = split(Lp[g][t]) (once per context), through a 32 x 32 LDS transpose.
__device__ __forceinline__ void k_lt_split_body(const uint3 bid_, const uint3 gdim_, const double* Lp, u16* hi, u16* lo, int64_t T, int G, int Gp) {
  __shared__ double tile[32][33];
  const int64_t t0 = (int64_t)bid_.x * 32;
  const int g0 = bid_.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int r = ty; r < 32; r += 8) {
    const int g = g0 + r;
    const int64_t t = t0 + tx;
    tile[r][tx] = (g < G && t < T) ? Lp[(int64_t)g * T + t] : 0.0;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int64_t t = t0 + r;
    const int g = g0 + tx;
    if (t < T && g < Gp) {
      u16 h, l;
      split_bf16(tile[tx][r], h, l);
      hi[t * Gp + g] = h;
      lo[t * Gp + g] = l;
    }
  }
}
struct F_k_lt_split {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_lt_split_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_lt_split(const double* Lp, u16* hi, u16* lo, int64_t T, int G, int Gp) {
  k_lt_split_body(blockIdx3(), gridDim3(), Lp, hi, lo, T, G, Gp);
}
void launch_lt_split(const DevState& s, hipStream_t st) {
  afq::glaunch<F_k_lt_split>(k_lt_split, dim3((unsigned)cdivu(s.T, 32), (unsigned)cdivu(s.Gp, 32)), dim3(256), 0, st, s.Lp,
                     s.Lt_hi, s.Lt_lo, s.T, s.G, s.Gp);
}

// Fb[w][c][g] = split(fields[w][g][c])
__device__ __forceinline__ void k_fields_split_body(const uint3 bid_, const uint3 gdim_, const double* fields, u16* hi, u16* lo, int W, int G, int Gp) {
  const int64_t total = (int64_t)W * 2 * Gp;
  for (int64_t e = (int64_t)bid_.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gdim_.x * blockDim.x) {
    const int g = (int)(e % Gp);
    const int64_t q = e / Gp;
    const double x = g < G ? fields[(q >> 1) * 2 * G + 2 * g + (q & 1)] : 0.0;
    u16 h, l;
    split_bf16(x, h, l);
    hi[e] = h;
    lo[e] = l;
  }
}
struct F_k_fields_split {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_fields_split_body(b, g, a...);
  }
};
__global__ void k_fields_split(const double* fields, u16* hi, u16* lo, int W, int G, int Gp) {
  k_fields_split_body(blockIdx3(), gridDim3(), fields, hi, lo, W, G, Gp);
}

// P[w][c] (both triangles) = sum_g field[w][g][c] L_g from the split operands.  A
// tile's 128 columns are a 16 x 8 block of V (rows i0.., orbitals j0..; blk lists the
// blocks that touch the lower triangle), each column reading the packed row of L_ij
// for j <= i, so the epilogue knows (i, j) without inverting the packed index and
// writes runs of 8 orbitals.  With Vh != nullptr the result goes straight to the split
// [-P_im | P_re] chunks that the split-BF16 Taylor series reads (Vh/Vl[w][chunk][i][32])
// instead of the FP64 P.  The tile is Eng::BM (walker, component) rows by one block;
// VHS_TILE 0: 128 rows, 64-deep single-buffered stages, two workgroups per CU; 1: 256
// rows, eight waves, 32-deep double-buffered stages (each block of L read by half as
// many tiles); 2: 128 rows, 32-deep double-buffered stages.
// VEC: the split output of the blocks below the diagonal staged through LDS and written
// as 16-byte runs (tiles 3 and 4: the GEMMs of tiles 0 and 2)
template <int VT> struct VhsTile;
template <> struct VhsTile<0> {
  template <int NS> using E = MmaBF16<128, 128, 2, 2, NS, NS, 64, false, true>;
  static constexpr int OCC = 2;
  static constexpr bool VEC = false;
};
template <> struct VhsTile<1> {
  template <int NS> using E = MmaBF16<256, 128, 4, 2, NS, NS, 32, true>;
  static constexpr int OCC = 1;
  static constexpr bool VEC = false;
};
template <> struct VhsTile<2> {
  template <int NS> using E = MmaBF16<128, 128, 2, 2, NS, NS, 32, true>;
  static constexpr int OCC = 2;
  static constexpr bool VEC = false;
};
template <> struct VhsTile<3> : VhsTile<0> { static constexpr bool VEC = true; };
template <> struct VhsTile<4> : VhsTile<2> { static constexpr bool VEC = true; };
constexpr int VHS_STG = 132;   // floats per staged row of the vectorized epilogue (128 + 4 against bank conflicts)
template <int NS, int VT>
__device__ __forceinline__ void k_vhs_bf16_body(const uint3 bid_, const uint3 gdim_, 
    const u16* Fh, const u16* Fl, const u16* Lh, const u16* Ll, double* P, const double* weights, int W,
    const int2* blk, int nblk, int N, int Gp, int gridx, int gridy, u16* Vh, u16* Vl, int Nq) {
  using Eng = typename VhsTile<VT>::template E<NS>;
  constexpr int BM = Eng::BM_, BPT = Eng::BN_ / 128;   // (walker, component) rows; blocks of V per tile
  __shared__ __attribute__((aligned(16))) unsigned char lds[Eng::LDS_BYTES];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, 1, 8);
  const int row0 = tl.y * BM;
  int2 bb[BPT];
#pragma unroll
  for (int q = 0; q < BPT; ++q) bb[q] = BPT * tl.x + q < nblk ? blk[BPT * tl.x + q] : int2{N, 0};   // i0 = N: no block
  bool any = false;
  for (int q = row0; q < min(row0 + BM, 2 * W); q += 2) any |= weights[q >> 1] > 1e-8;
  if (!any) return;
  Eng e;
  e.run(
      [&](int c, int r) -> const u16* {
        const int q = row0 + r;
        return q < 2 * W ? (c ? Fl : Fh) + (int64_t)q * Gp : nullptr;
      },
      [&](int c, int col) -> const u16* {
        const int2 b0 = bb[col >> 7];
        const int i = b0.x + ((col & 127) >> 3), j = b0.y + (col & 7);
        if (i >= N || j > i) return nullptr;
        return (c ? Ll : Lh) + ((int64_t)i * (i + 1) / 2 + j) * Gp;
      },
      Gp, lds);
  // (the staging needs the LDS of the split engine; the one-pass form keeps the scalar stores)
  if constexpr (VhsTile<VT>::VEC && Eng::LDS_BYTES >= BM * VHS_STG * 4) {
    // A block of V strictly below the diagonal (every j < every i): its split values go
    // out as 16-byte runs.  The run() above ends with a barrier, so the staging may reuse
    // the operand LDS.  V[i][j] for the block's 8 j's is a run of 8 in row (w, j0/16, i);
    // V[j][i] for its 16 i's is the run of 16 in row (w, i0/16, j).  Entries past N are
    // zero (their L rows load as zero), as the zero pads of the layout need; rows past N
    // are not written.
    static_assert(BPT == 1, "one block of V per tile");
    const int i0 = bb[0].x, j0 = bb[0].y;
    if (Vh && j0 + 7 < i0) {
      float* stg = reinterpret_cast<float*>(lds);
      e.store([&](int r, int c, float v) { stg[r * VHS_STG + c] = v; });
      __syncthreads();
      const int64_t wstride = (int64_t)(Nq >> 4) * N * 32;
      auto split8 = [](const float* x, bool neg, uint4& h, uint4& l) {
        float a[4], b[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          a[k] = neg ? -x[k] : x[k];
          b[k] = neg ? -x[k + 4] : x[k + 4];
        }
        uint2 ha, la, hb, lb;
        split4_bf16(a, ha, la);
        split4_bf16(b, hb, lb);
        h = make_uint4(ha.x, ha.y, hb.x, hb.y);
        l = make_uint4(la.x, la.y, lb.x, lb.y);
      };
      // V[i][j]: (walker, i, component) -> 8 values
      for (int u = threadIdx.x; u < BM * 16; u += Eng::NT) {
        const int comp = u & 1, ii = (u >> 1) & 15, wl = u >> 5;
        const int q = 2 * wl + comp, i = i0 + ii;
        if (row0 + q >= 2 * W || i >= N) continue;
        float x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = stg[q * VHS_STG + ii * 8 + k];
        uint4 h, l;
        split8(x, comp != 0, h, l);
        const int64_t o = ((row0 + q) >> 1) * wstride + ((int64_t)(j0 >> 4) * N + i) * 32 + (comp ? 0 : 16) + (j0 & 15);
        *reinterpret_cast<uint4*>(Vh + o) = h;
        *reinterpret_cast<uint4*>(Vl + o) = l;
      }
      // V[j][i]: (walker, j, component) -> 16 values
      for (int u = threadIdx.x; u < BM * 8; u += Eng::NT) {
        const int comp = u & 1, jj = (u >> 1) & 7, wl = u >> 4;
        const int q = 2 * wl + comp, j = j0 + jj;
        if (row0 + q >= 2 * W || j >= N) continue;
        const int64_t o = ((row0 + q) >> 1) * wstride + ((int64_t)(i0 >> 4) * N + j) * 32 + (comp ? 0 : 16);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          float x[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) x[k] = stg[q * VHS_STG + (half * 8 + k) * 8 + jj];
          uint4 h, l;
          split8(x, comp != 0, h, l);
          *reinterpret_cast<uint4*>(Vh + o + half * 8) = h;
          *reinterpret_cast<uint4*>(Vl + o + half * 8) = l;
        }
      }
      return;
    }
  }
  e.store([&](int r, int c, float v) {
    const int q = row0 + r;
    const int2 b0 = bb[c >> 7];
    const int i = b0.x + ((c & 127) >> 3), j = b0.y + (c & 7);
    if (q >= 2 * W || i >= N || j > i) return;
    if (Vh) {
      const int w = q >> 1, comp = q & 1;
      const float x = comp ? -v : v;
      const u16 h = f2bf_bits(x), l = f2bf_bits(x - bf_bits2f(h));
      const int64_t base = (int64_t)w * (Nq >> 4) * N * 32;
      const int off = comp ? 0 : 16;
      const int64_t e1 = base + ((int64_t)(j >> 4) * N + i) * 32 + off + (j & 15);
      const int64_t e2 = base + ((int64_t)(i >> 4) * N + j) * 32 + off + (i & 15);
      Vh[e1] = h; Vl[e1] = l;
      Vh[e2] = h; Vl[e2] = l;
      return;
    }
    double* Pq = P + (int64_t)q * N * N;
    Pq[(int64_t)i * N + j] = (double)v;
    Pq[(int64_t)j * N + i] = (double)v;
  });
}
template <int NS, int VT>
struct F_k_vhs_bf16 {
  static constexpr int NT = VhsTile<VT>::template E<NS>::NT, OCC = VhsTile<VT>::OCC;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_vhs_bf16_body<NS, VT>(b, g, a...);
  }
};
template <int NS, int VT>
__global__ __launch_bounds__(VhsTile<VT>::template E<NS>::NT, VhsTile<VT>::OCC) void k_vhs_bf16(
    const u16* Fh, const u16* Fl, const u16* Lh, const u16* Ll, double* P, const double* weights, int W,
    const int2* blk, int nblk, int N, int Gp, int gridx, int gridy, u16* Vh, u16* Vl, int Nq) {
  k_vhs_bf16_body<NS, VT>(blockIdx3(), gridDim3(), Fh, Fl, Lh, Ll, P, weights, W, blk, nblk, N, Gp, gridx, gridy, Vh, Vl, Nq);
}

void launch_vhs_lp(const DevState& s, int prec, hipStream_t st) {
  const int64_t tot = (int64_t)s.W * 2 * s.Gp;
  afq::glaunch<F_k_fields_split>(k_fields_split, dim3((unsigned)std::min<int64_t>(cdivu(tot, 256), 65535)), dim3(256), 0, st,
                     s.fields, s.Fb_hi, s.Fb_lo, s.W, s.G, s.Gp);
  u16* vh = s.prec_prop != AFQ_PREC_FP64 ? s.Vh : nullptr;
  u16* vl = s.prec_prop != AFQ_PREC_FP64 ? s.Vl : nullptr;
  const int2* blk = reinterpret_cast<const int2*>(s.vhs_blk);
  auto go = [&](auto ns, auto vt) {
    constexpr int NS = decltype(ns)::value, VT = decltype(vt)::value;
    using Eng = typename VhsTile<VT>::template E<NS>;
    const int gx = (int)cdivu(s.nvhs_blk, Eng::BN_ / 128), gy = (int)cdivu(2 * (int64_t)s.W, Eng::BM_);
    afq::glaunch<F_k_vhs_bf16<NS, VT>>((k_vhs_bf16<NS, VT>), dim3(gx * gy), dim3(Eng::NT), 0, st, s.Fb_hi, s.Fb_lo, s.Lt_hi, s.Lt_lo,
                       s.P, s.weights, s.W, blk, s.nvhs_blk, s.N, s.Gp, gx, gy, vh, vl, s.Nq);
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  using I4 = std::integral_constant<int, 4>;
  const int vt = s.vhs_tile;
  if (prec == AFQ_PREC_BF16X3) {
    if (vt == 1) go(I2{}, I1{});
    else if (vt == 2) go(I2{}, I2{});
    else if (vt == 3) go(I2{}, I3{});
    else if (vt == 4) go(I2{}, I4{});
    else go(I2{}, std::integral_constant<int, 0>{});
  } else {
    if (vt == 1) go(I1{}, I1{});
    else if (vt == 2) go(I1{}, I2{});
    else if (vt == 3) go(I1{}, I3{});
    else if (vt == 4) go(I1{}, I4{});
    else go(I1{}, std::integral_constant<int, 0>{});
  }
}

// E_L = ecore + sum_s m_s e1_s + 1/2 sum_{g<GE} fb_g^2 - 1/2 sum_s m_s X_s
__device__ __forceinline__ void k_energy_body(const uint3 bid_, const uint3 gdim_, const double* fb, const double* e1, const double* Xp,
                                               const double* logO, const double* weights, const int* sel,
                                               double* eloc, double* ho, int G, int GE, int W, int nslots,
                                               int m0, int m1, int ngt_used0, int ngt_used1, int ngt_cap,
                                               double ecore, double delta) {
  const int idx = bid_.x;
  const int w = sel ? sel[idx] : idx;
  const int lane = threadIdx.x;
  double jr = 0.0, ji = 0.0;
  for (int g = lane; g < GE; g += 64) {
    const double a = fb[(int64_t)w * 2 * G + 2 * g], b = fb[(int64_t)w * 2 * G + 2 * g + 1];
    jr += a * a - b * b;
    ji += 2.0 * a * b;
  }
  double xr = 0.0, xi = 0.0;
  for (int s = 0; s < nslots; ++s) {
    const int m = s == 0 ? m0 : m1, nt = s == 0 ? ngt_used0 : ngt_used1;
    for (int t = lane; t < nt; t += 64) {
      const double* o = Xp + 2 * (((int64_t)s * W + w) * ngt_cap + t);
      xr += m * o[0];
      xi += m * o[1];
    }
  }
  jr = wave_sum(jr); ji = wave_sum(ji); xr = wave_sum(xr); xi = wave_sum(xi);
  if (lane == 0) {
    double er = ecore, ei = 0.0;
    for (int s = 0; s < nslots; ++s) {
      const int m = s == 0 ? m0 : m1;
      er += m * e1[2 * ((int64_t)w * nslots + s)];
      ei += m * e1[2 * ((int64_t)w * nslots + s) + 1];
    }
    er += 0.5 * (jr - xr);
    ei += 0.5 * (ji - xi);
    const bool live = weights == nullptr || weights[w] != 0.0;
    eloc[w] = live ? er + delta : 0.0;
    if (ho) {
      const cplx O = cexp(cplx{logO[2 * w], logO[2 * w + 1]});
      const cplx EO = live ? cmul(cplx{er, ei}, O) : cplx{0.0, 0.0};  // dead: no exchange was computed
      ho[4 * w] = EO.re; ho[4 * w + 1] = EO.im; ho[4 * w + 2] = O.re; ho[4 * w + 3] = O.im;
    }
  }
}
struct F_k_energy {
  static constexpr int NT = 64, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_energy_body(b, g, a...);
  }
};
__global__ __launch_bounds__(64) void k_energy(const double* fb, const double* e1, const double* Xp,
                                               const double* logO, const double* weights, const int* sel,
                                               double* eloc, double* ho, int G, int GE, int W, int nslots,
                                               int m0, int m1, int ngt_used0, int ngt_used1, int ngt_cap,
                                               double ecore, double delta) {
  k_energy_body(blockIdx3(), gridDim3(), fb, e1, Xp, logO, weights, sel, eloc, ho, G, GE, W, nslots, m0, m1, ngt_used0, ngt_used1, ngt_cap, ecore, delta);
}

void launch_energy(const DevState& s, const int* sel, int nsel, double delta, hipStream_t st) {
  const int ng0 = (int)cdivu(s.GE, exchange_tile_g(s.slot[0].n));
  const int ng1 = s.nslots > 1 ? (int)cdivu(s.GE, exchange_tile_g(s.slot[1].n)) : 0;
  afq::glaunch<F_k_energy>(k_energy, dim3(nsel), dim3(64), 0, st, s.fb, s.e1, s.Xp, s.logO, s.weights, sel, s.eloc,
                     s.ho, s.G, s.GE, s.W, s.nslots, s.slot[0].mult, s.nslots > 1 ? s.slot[1].mult : 0, ng0,
                     ng1, s.ngt_cap, s.ecore, delta);
}

// ------------------------------------------------------------------ one-body density matrix
// Mixed-estimator 1-RDM (DQMC/MixedEstimator.cpp:492-510): the weighted sum over
// walkers of Re(G_s^T) = Phi_s Re(theta_s)^T needs only sum_w w Re(theta_s[w])
// (Phi_s is real).  Element e < Ktot of a walker's theta carries that sum; element
// Ktot carries sum_w w.  Pass 1: RDM_CH fixed chunks of walkers each add their
// walkers of nonzero weight in ascending order into part[ch][e]; pass 2 adds the
// chunks in order into acc[e], so the sums do not depend on scheduling.  Walkers
// of weight zero are not read (their theta is not kept current).
constexpr int RDM_CH = 32;
__device__ __forceinline__ void k_rdm_part_body(const uint3 bid_, const uint3 gdim_, const double* __restrict__ theta,
                                                  const double* __restrict__ weights, int W, int64_t Ktot,
                                                  double* __restrict__ part) {
  const int64_t e = (int64_t)bid_.x * blockDim.x + threadIdx.x;
  if (e > Ktot) return;
  const int per = (W + RDM_CH - 1) / RDM_CH;
  const int w0 = bid_.y * per, w1 = min(W, w0 + per);
  double s = 0.0;
  for (int w = w0; w < w1; ++w) {
    const double wt = weights[w];
    if (wt == 0.0) continue;
    s += wt * (e < Ktot ? theta[2 * ((int64_t)w * Ktot + e)] : 1.0);
  }
  part[(int64_t)bid_.y * (Ktot + 1) + e] = s;
}
struct F_k_rdm_part {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_rdm_part_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_rdm_part(const double* __restrict__ theta,
                                                  const double* __restrict__ weights, int W, int64_t Ktot,
                                                  double* __restrict__ part) {
  k_rdm_part_body(blockIdx3(), gridDim3(), theta, weights, W, Ktot, part);
}
__device__ __forceinline__ void k_rdm_add_body(const uint3 bid_, const uint3 gdim_, const double* __restrict__ part, double* __restrict__ acc,
                                                 int64_t n) {
  const int64_t e = (int64_t)bid_.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  double s = acc[e];
  for (int ch = 0; ch < RDM_CH; ++ch) s += part[(int64_t)ch * n + e];
  acc[e] = s;
}
struct F_k_rdm_add {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_rdm_add_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_rdm_add(const double* __restrict__ part, double* __restrict__ acc,
                                                 int64_t n) {
  k_rdm_add_body(blockIdx3(), gridDim3(), part, acc, n);
}
int64_t rdm_part_doubles(const DevState& s) { return (int64_t)RDM_CH * (s.Ktot + 1); }
void launch_rdm_accumulate(const DevState& s, double* part, double* acc, hipStream_t st) {
  const int64_t n = s.Ktot + 1;
  const unsigned bx = (unsigned)cdivu(n, 256);
  afq::glaunch<F_k_rdm_part>(k_rdm_part, dim3(bx, RDM_CH), dim3(256), 0, st, s.theta, s.weights, s.W, s.Ktot, part);
  afq::glaunch<F_k_rdm_add>(k_rdm_add, dim3(bx), dim3(256), 0, st, part, acc, n);
}

// ------------------------------------------------------------------ comb
// Sequential cumulative sum, exactly the reference's order (DQMC/MixedEstimator.cpp:595-598).
// The block stages chunks of the weights through LDS with coalesced loads; one thread
// runs the dependent additions out of LDS, in order, carrying the sum across chunks.
constexpr int CUMSUM_CHUNK = 4096;
// c + v[0] + v[1] + .. + v[n - 1], added in that order by one lane, f(i, sum) after each: 16
// elements are read ahead of the chain of additions, so that an element costs an addition and not
// an LDS read's latency too (1024 elements 12.6 us, now 10.3).
template <class F>
__device__ __forceinline__ double chain_sum(const double* v, int n, double c, const F& f) {
  constexpr int U = 16;
  double a[U], b[U];
  const int m = n / U * U;
  auto get = [&](double (&r)[U], int i) {
#pragma unroll
    for (int q = 0; q < U; ++q) r[q] = v[i + q];
  };
  auto add = [&](const double (&r)[U], int i) {
#pragma unroll
    for (int q = 0; q < U; ++q) {
      c += r[q];
      f(i + q, c);
    }
  };
  int i = 0;
  if (m > 0) get(a, 0);
  for (; i + U < m; i += 2 * U) {
    get(b, i + U);
    add(a, i);
    if (i + 2 * U < m) get(a, i + 2 * U);
    add(b, i + U);
  }
  if (i < m) {
    add(a, i);
    i += U;
  }
  for (; i < n; ++i) {
    c += v[i];
    f(i, c);
  }
  return c;
}
__device__ __forceinline__ void k_cumsum_body(const uint3 bid_, const uint3 gdim_, const double* __restrict__ w, double* __restrict__ cum, int W) {
  __shared__ double buf[CUMSUM_CHUNK];
  double c = 0.0;  // the running sum, kept by thread 0
  for (int base = 0; base < W; base += CUMSUM_CHUNK) {
    const int n = min(CUMSUM_CHUNK, W - base);
    for (int i = threadIdx.x; i < n; i += blockDim.x) buf[i] = w[base + i];
    __syncthreads();
    if (threadIdx.x == 0) c = chain_sum(buf, n, base == 0 ? -0.0 : c, [&](int i, double x) { buf[i] = x; });   // -0 + x is x
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) cum[base + i] = buf[i];
    __syncthreads();
  }
}
struct F_k_cumsum {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_cumsum_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_cumsum(const double* __restrict__ w, double* __restrict__ cum, int W) {
  k_cumsum_body(blockIdx3(), gridDim3(), w, cum, W);
}
__device__ __forceinline__ void k_comb_index_body(const uint3 bid_, const uint3 gdim_, const double* cum, int* idx, double* weights, int W, double zeta,
                             const double* zeta_dev, double* st) {
  const int w = bid_.x * blockDim.x + threadIdx.x;
  if (w >= W) return;
  if (zeta_dev) zeta = *zeta_dev;
  const double tot = cum[W - 1];
  const double z = (w + zeta) / W;
  const double target = z * tot;
  int lo = 0, hi = W;  // lower_bound
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (cum[mid] < target) lo = mid + 1; else hi = mid;
  }
  idx[w] = lo < W ? lo : W - 1;
  weights[w] = tot / W;
  if (w == 0 && st) st[SS_COMB] = tot;
}
struct F_k_comb_index {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_comb_index_body(b, g, a...);
  }
};
__global__ void k_comb_index(const double* cum, int* idx, double* weights, int W, double zeta,
                             const double* zeta_dev, double* st) {
  k_comb_index_body(blockIdx3(), gridDim3(), cum, idx, weights, W, zeta, zeta_dev, st);
}
// The comb's copies of every per-walker array in one launch: dst[w] = src[idx[w]].  A captured step
// gathers into the spare buffers and copies back (back: src and dst change places), so that every
// replay finds the walkers where its nodes expect them; a walker that stays where it is is then
// left alone in both.  per: doubles a walker, even.  One launch for four or five arrays instead of
// one each (and one for the new weights) takes 9 launches out of a block of five steps at N = 10:
// 310 -> 292 us of kernels; a captured step of 24 systems goes from 204 launches to 164.
struct GatherArgs {
  const int* idx;
  double *src[5], *dst[5];
  int64_t per[5];
  int narr, skip, back;
};
__device__ __forceinline__ void k_gather_body(const uint3 bid_, const uint3 gdim_, const GatherArgs a) {
  const int w = bid_.y, from = a.idx[w];
  if (a.skip && from == w) return;
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    if (q >= a.narr) break;
    const int64_t n = a.per[q] / 2;
    const double2* s = reinterpret_cast<const double2*>(a.back ? a.dst[q] : a.src[q]) + (a.back ? w : from) * n;
    double2* d = reinterpret_cast<double2*>(a.back ? a.src[q] : a.dst[q]) + w * n;
    for (int64_t i = (int64_t)bid_.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gdim_.x * blockDim.x) d[i] = s[i];
  }
}
struct F_k_gather {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_gather_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_gather(const GatherArgs a) {
  k_gather_body(blockIdx3(), gridDim3(), a);
}

// plain streaming copy (read n, write n doubles): the HBM-traffic calibration kernel
__device__ __forceinline__ void k_copy_calib_body(const uint3 bid_, const uint3 gdim_, const double* __restrict__ a, double* __restrict__ b, int64_t n) {
  for (int64_t i = (int64_t)bid_.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gdim_.x * blockDim.x)
    b[i] = a[i];
}
struct F_k_copy_calib {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_copy_calib_body(b, g, a...);
  }
};
__global__ void k_copy_calib(const double* __restrict__ a, double* __restrict__ b, int64_t n) {
  k_copy_calib_body(blockIdx3(), gridDim3(), a, b, n);
}

// Block totals of one population: out = {sum w, sum w clip(E_L), walkers propagated
// in the step, walkers of nonzero weight} over the live walkers, the clip to
// center -+ halfw of DQMC/MixedEstimator.cpp:525-530 (none when center is null);
// cnt[1] is the weight kernel's count of the walkers it propagated.
__device__ __forceinline__ void k_block_energy_body(const uint3 bid_, const uint3 gdim_, const double* eloc, const double* weights, int W,
                                                      const double* center, double halfw,
                                                      const unsigned long long* cnt, double* out) {
  __shared__ double red[16];
  double sw = 0.0, swe = 0.0, nl = 0.0;
  const double c0 = center ? *center : 0.0;
  for (int w = threadIdx.x; w < W; w += blockDim.x) {
    const double wt = weights[w];
    if (wt != 0.0) {
      double e = eloc[w];
      if (center) e = fmin(fmax(e, c0 - halfw), c0 + halfw);
      sw += wt;
      swe += wt * e;
      nl += 1.0;
    }
  }
  sw = block_sum(sw, red);
  swe = block_sum(swe, red);
  nl = block_sum(nl, red);
  if (threadIdx.x == 0) {
    out[0] = sw;
    out[1] = swe;
    out[2] = cnt ? (double)cnt[1] : 0.0;
    out[3] = nl;
  }
}
struct F_k_block_energy {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_block_energy_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_block_energy(const double* eloc, const double* weights, int W,
                                                      const double* center, double halfw,
                                                      const unsigned long long* cnt, double* out) {
  k_block_energy_body(blockIdx3(), gridDim3(), eloc, weights, W, center, halfw, cnt, out);
}
void launch_block_energy(const DevState& s, const double* center, double halfw, double* out, hipStream_t st) {
  afq::glaunch<F_k_block_energy>(k_block_energy, dim3(1), dim3(256), 0, st, s.eloc, s.weights, s.W, center, halfw,
                     (const unsigned long long*)s.ncap, out);
}

// ------------------------------------------------------------------ population statistics
// The per-step numbers the driver's population control reads (DQMC/MixedEstimator.cpp:
// 461-475, 513-538), kept in the context's small device array st (StatSlot order) so a
// step needs one small copy to the host.  Sums over walkers run in walker order on one
// thread, as the reference's rank-0 loops do, so the totals are the same bits as a
// host loop over the same weights.

// st[SS_SUMW] = sum of the weights, st[SS_NLIVE] = walkers of nonzero weight, and the
// step counters (capped, propagated)
__device__ __forceinline__ void k_step_stats_body(const uint3 bid_, const uint3 gdim_, const double* __restrict__ w, int W,
                                                    const unsigned long long* cnt, double* st) {
  __shared__ double buf[CUMSUM_CHUNK];
  __shared__ double red[16];
  double sum = 0.0, nl = 0.0;
  for (int base = 0; base < W; base += CUMSUM_CHUNK) {
    const int n = min(CUMSUM_CHUNK, W - base);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      const double x = w[base + i];
      buf[i] = x;
      nl += x != 0.0 ? 1.0 : 0.0;
    }
    __syncthreads();
    if (threadIdx.x == 0) sum = chain_sum(buf, n, sum, [](int, double) {});
    __syncthreads();
  }
  nl = block_sum(nl, red);
  if (threadIdx.x == 0) {
    st[SS_SUMW] = sum;
    st[SS_NLIVE] = nl;
    st[SS_NCAP] = cnt ? (double)cnt[0] : 0.0;
    st[SS_NPROP] = cnt ? (double)cnt[1] : 0.0;
  }
}
struct F_k_step_stats {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_step_stats_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_step_stats(const double* __restrict__ w, int W,
                                                    const unsigned long long* cnt, double* st) {
  k_step_stats_body(blockIdx3(), gridDim3(), w, W, cnt, st);
}
void launch_step_stats(const DevState& s, hipStream_t st) {
  afq::glaunch<F_k_step_stats>(k_step_stats, dim3(1), dim3(256), 0, st, s.weights, s.W, s.ncap, s.stats);
}

// Block totals of the last measurement: every live walker's local energy, clipped to
// its rank's running average -+ halfw when clip is set (DQMC/MixedEstimator.cpp:525-530:
// |E - c| > halfw moves E to c -+ halfw), dead walkers' energies set to zero; eloc is
// rewritten with those values.  st receives sum w, sum w E (walker order), the variance
// of the weighted mean sum w^2 (E - m)^2 / (sum w)^2, and the counts of live, clipped and
// non-finite energies.
__device__ __forceinline__ void k_block_totals_body(const uint3 bid_, const uint3 gdim_, double* __restrict__ eloc, const double* __restrict__ w, int W,
                                                      const double* center, int nwr, double halfw, int clip,
                                                      double* st) {
  constexpr int CH = CUMSUM_CHUNK / 2;
  __shared__ double bw[CH], be[CH];
  __shared__ double red[16];
  __shared__ double mean;
  double sw = 0.0, swe = 0.0, nl = 0.0, nc = 0.0, nbad = 0.0;
  for (int base = 0; base < W; base += CH) {
    const int n = min(CH, W - base);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      const int q = base + i;
      const double wt = w[q];
      double e = eloc[q];
      if (wt == 0.0) {
        e = 0.0;
      } else {
        nl += 1.0;
        if (!isfinite(e)) {
          nbad += 1.0;
        } else if (clip) {
          const double c = center[q / nwr];
          if (fabs(e - c) > halfw) {
            nc += 1.0;
            e = e > c ? c + halfw : c - halfw;
          }
        }
      }
      eloc[q] = e;
      bw[i] = wt;
      be[i] = e;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      // product and sum rounded separately (no fused multiply-add), as the host loop does
#pragma clang fp contract(off)
      for (int i = 0; i < n; ++i) {
        sw += bw[i];
        const double p = be[i] * bw[i];
        swe += p;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) mean = swe / sw;
  __syncthreads();
  const double m = mean;
  double v = 0.0;
  for (int q = threadIdx.x; q < W; q += blockDim.x) {
    const double wt = w[q], d = eloc[q] - m;
    v += wt * wt * d * d;
  }
  v = block_sum(v, red);
  nl = block_sum(nl, red);
  nc = block_sum(nc, red);
  nbad = block_sum(nbad, red);
  if (threadIdx.x == 0) {
    st[SS_BW] = sw;
    st[SS_BWE] = swe;
    st[SS_BVAR] = v / (sw * sw);
    st[SS_NMEAS] = nl;
    st[SS_NCLIP] = nc;
    st[SS_NBAD] = nbad;
  }
}
struct F_k_block_totals {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_block_totals_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_block_totals(double* __restrict__ eloc, const double* __restrict__ w, int W,
                                                      const double* center, int nwr, double halfw, int clip,
                                                      double* st) {
  k_block_totals_body(blockIdx3(), gridDim3(), eloc, w, W, center, nwr, halfw, clip, st);
}
void launch_block_totals(const DevState& s, const double* center, int nwr, double halfw, bool clip,
                         double* st_out, hipStream_t st) {
  afq::glaunch<F_k_block_totals>(k_block_totals, dim3(1), dim3(256), 0, st, s.eloc, s.weights, s.W, center, nwr, halfw,
                     (int)(clip && center && halfw > 0.0), st_out);
}

// every walker's orbitals = the determinant at src (one walker's serial block)
__device__ __forceinline__ void k_broadcast_det_body(const uint3 bid_, const uint3 gdim_, double* __restrict__ psi, const double* __restrict__ src, int64_t per) {
  double* d = psi + (int64_t)bid_.y * per;
  for (int64_t i = (int64_t)bid_.x * blockDim.x + threadIdx.x; i < per; i += (int64_t)gdim_.x * blockDim.x)
    d[i] = src[i];
}
struct F_k_broadcast_det {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_broadcast_det_body(b, g, a...);
  }
};
__global__ void k_broadcast_det(double* __restrict__ psi, const double* __restrict__ src, int64_t per) {
  k_broadcast_det_body(blockIdx3(), gridDim3(), psi, src, per);
}
void launch_broadcast_det(const DevState& s, const double* src, hipStream_t st) {
  const int64_t per = 2 * s.ms;
  const unsigned bx = (unsigned)std::min<int64_t>(64, (per + 255) / 256);
  afq::glaunch<F_k_broadcast_det>(k_broadcast_det, dim3(bx, s.W), dim3(256), 0, st, s.psi, src, per);
}

__device__ __forceinline__ void k_step_inc_body(const uint3 bid_, const uint3 gdim_, unsigned long long* step) {
  if (threadIdx.x == 0 && bid_.x == 0) *step += 1ull;
}
struct F_k_step_inc {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_step_inc_body(b, g, a...);
  }
};
__global__ void k_step_inc(unsigned long long* step) {
  k_step_inc_body(blockIdx3(), gridDim3(), step);
}
void launch_step_inc(unsigned long long* step, hipStream_t st) {
  afq::glaunch<F_k_step_inc>(k_step_inc, dim3(1), dim3(64), 0, st, step);
}

void launch_comb(DevState& s, double zeta, hipStream_t st) {
  s.tb_live = false;
  s.tb_post = false;
  afq::glaunch<F_k_cumsum>(k_cumsum, dim3(1), dim3(256), 0, st, s.weights, s.cum, s.W);
  afq::glaunch<F_k_comb_index>(k_comb_index, dim3(cdivu(s.W, 256)), dim3(256), 0, st, s.cum, s.idx, s.weights, s.W, zeta,
                     s.d_zeta, s.stats);
  GatherArgs g{};
  g.idx = s.idx;
  auto add = [&](double*& a, double*& b, int64_t per) {
    g.src[g.narr] = a;
    g.dst[g.narr] = b;
    g.per[g.narr++] = per;
    if (!s.graph_mode) std::swap(a, b);
  };
  add(s.psi, s.psi2, 2 * s.ms);
  if (s.graph_mode) add(s.theta, s.theta2, 2 * s.Ktot);
  else s.theta_stale = true;
  add(s.fb, s.fb2, 2 * (int64_t)s.G);
  add(s.logO, s.logO2, 2);
  add(s.e1, s.e12, 2 * (int64_t)s.nslots);
  const unsigned bx = (unsigned)std::min<int64_t>(64, std::max(s.ms, (int64_t)s.G) / 256 + 1);
  g.skip = s.graph_mode;
  afq::glaunch<F_k_gather>(k_gather, dim3(bx, s.W), dim3(256), 0, st, g);
  if (s.graph_mode) {
    g.back = 1;
    afq::glaunch<F_k_gather>(k_gather, dim3(bx, s.W), dim3(256), 0, st, g);
  }
}

__device__ __forceinline__ void k_copy_det0_body(const uint3 bid_, const uint3 gdim_, double* dst, const double* src, int64_t ms, int64_t n0, int64_t off1) {
  const int w = bid_.y;
  for (int64_t i = (int64_t)bid_.x * blockDim.x + threadIdx.x; i < 2 * n0; i += (int64_t)gdim_.x * blockDim.x)
    dst[2 * (w * ms + off1) + i] = src[2 * w * ms + i];
}
struct F_k_copy_det0 {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_copy_det0_body(b, g, a...);
  }
};
__global__ void k_copy_det0(double* dst, const double* src, int64_t ms, int64_t n0, int64_t off1) {
  k_copy_det0_body(blockIdx3(), gridDim3(), dst, src, ms, n0, off1);
}
void launch_copy_det0_to_det1(const DevState& s, double* dst, const double* src, hipStream_t st) {
  const int64_t n0 = (int64_t)s.N * s.det_n[0];
  afq::glaunch<F_k_copy_det0>(k_copy_det0, dim3(cdivu(2 * n0, 256), s.W), dim3(256), 0, st, dst, src, s.ms, n0,
                     s.det_off[1]);
}

// ------------------------------------------------------------------ Hamiltonian setup
// floattenCholesky layout (DQMC/Hamiltonian.cpp:179-220): Lp[g][i(i+1)/2 + j], j <= i
__device__ __forceinline__ void k_pack_chol_body(const uint3 bid_, const uint3 gdim_, const double* L, double* Lp, int N, int G, int64_t T, int round_f32) {
  const int g = bid_.y;
  for (int64_t t = (int64_t)bid_.x * blockDim.x + threadIdx.x; t < T; t += (int64_t)gdim_.x * blockDim.x) {
    // invert t = i(i+1)/2 + j
    int i = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while ((int64_t)(i + 1) * (i + 2) / 2 <= t) ++i;
    while ((int64_t)i * (i + 1) / 2 > t) --i;
    const int j = (int)(t - (int64_t)i * (i + 1) / 2);
    const double v = L[(int64_t)g * N * N + (int64_t)i * N + j];
    Lp[(int64_t)g * T + t] = round_f32 ? (double)(float)v : v;
  }
}
struct F_k_pack_chol {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_pack_chol_body(b, g, a...);
  }
};
__global__ void k_pack_chol(const double* L, double* Lp, int N, int G, int64_t T, int round_f32) {
  k_pack_chol_body(blockIdx3(), gridDim3(), L, Lp, N, G, T, round_f32);
}
void launch_pack_chol(const double* L, double* Lp, int N, int G, int64_t T, bool round_f32, hipStream_t st) {
  afq::glaunch<F_k_pack_chol>(k_pack_chol, dim3((unsigned)std::min<int64_t>(256, (T + 255) / 256), G), dim3(256), 0, st, L,
                     Lp, N, G, T, (int)round_f32);
}

// rotateCholesky (DQMC/Hamiltonian.cpp:52-133): R[g][koff + k*n + i] = sum_m Phi(m,i) L_g(m,k)
constexpr int RC_BM = 64, RC_BN = 128;
__device__ __forceinline__ void k_rotate_chol_body(const uint3 bid_, const uint3 gdim_, const double* L, const double* phi, double* R, int N, int n,
                                                     int G, int64_t Ktot, int64_t koff) {
  using Eng = MmaF64<RC_BM, RC_BN, 2, 2, true, true>;
  __shared__ double lds[Eng::LDS_DOUBLES];
  const int64_t ncol = (int64_t)G * N;
  const int64_t q0 = (int64_t)bid_.x * RC_BN;
  const int row0 = bid_.y * RC_BM;
  Eng e;
  e.run([&](int r, int m) { const int i = row0 + r; return (i < n && m < N) ? phi[(int64_t)m * n + i] : 0.0; },
        [&](int m, int c) {
          const int64_t q = q0 + c;
          if (q >= ncol || m >= N) return 0.0;
          const int64_t g = q / N, k = q - g * N;
          return L[g * N * N + (int64_t)m * N + k];
        },
        N, lds);
  e.store([&](int r, int c, double v) {
    const int i = row0 + r;
    const int64_t q = q0 + c;
    if (i >= n || q >= ncol) return;
    const int64_t g = q / N, k = q - g * N;
    R[g * Ktot + koff + k * n + i] = v;
  });
}
struct F_k_rotate_chol {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_rotate_chol_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_rotate_chol(const double* L, const double* phi, double* R, int N, int n,
                                                     int G, int64_t Ktot, int64_t koff) {
  k_rotate_chol_body(blockIdx3(), gridDim3(), L, phi, R, N, n, G, Ktot, koff);
}
void launch_rotate_chol(const double* L, const double* phi, double* R, int N, int n, int G, int64_t Ktot,
                        int64_t koff, hipStream_t st) {
  dim3 grid(cdivu((int64_t)G * N, RC_BN), cdivu(n, RC_BM));
  afq::glaunch<F_k_rotate_chol>(k_rotate_chol, grid, dim3(256), 0, st, L, phi, R, N, n, G, Ktot, koff);
}

// plain row-major C = A B through the tile engine (parity hook for the MFMA lane layout)
__device__ __forceinline__ void k_debug_gemm_body(const uint3 bid_, const uint3 gdim_, const double* A, const double* B, double* C, int M, int N, int K) {
  using Eng = MmaF64<64, 128, 2, 2, false, true>;
  __shared__ double lds[Eng::LDS_DOUBLES];
  const int r0 = bid_.y * 64, c0 = bid_.x * 128;
  Eng e;
  e.run([&](int r, int k) { return (r0 + r < M && k < K) ? A[(int64_t)(r0 + r) * K + k] : 0.0; },
        [&](int k, int c) { return (k < K && c0 + c < N) ? B[(int64_t)k * N + c0 + c] : 0.0; }, K, lds);
  e.store([&](int r, int c, double v) {
    if (r0 + r < M && c0 + c < N) C[(int64_t)(r0 + r) * N + c0 + c] = v;
  });
}
struct F_k_debug_gemm {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_debug_gemm_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_debug_gemm(const double* A, const double* B, double* C, int M, int N, int K) {
  k_debug_gemm_body(blockIdx3(), gridDim3(), A, B, C, M, N, K);
}
void launch_debug_gemm(const double* A, const double* B, double* C, int M, int N, int K, hipStream_t st) {
  afq::glaunch<F_k_debug_gemm>(k_debug_gemm, dim3(cdivu(N, 128), cdivu(M, 64)), dim3(256), 0, st, A, B, C, M, N, K);
}

// split an FP64 matrix M x K (row-major) into K-contiguous bf16 hi/lo rows with padded K
__device__ __forceinline__ void k_split_rows_body(const uint3 bid_, const uint3 gdim_, const double* X, u16* hi, u16* lo, int M, int K, int Kp, int transpose) {
  // transpose == 0: row m of X -> row m;  transpose == 1: X is K x M (row-major), column m -> row m
  const int64_t total = (int64_t)M * Kp;
  for (int64_t e = (int64_t)bid_.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gdim_.x * blockDim.x) {
    const int m = (int)(e / Kp), k = (int)(e % Kp);
    double x = 0.0;
    if (k < K) x = transpose ? X[(int64_t)k * M + m] : X[(int64_t)m * K + k];
    u16 h, l;
    split_bf16(x, h, l);
    hi[e] = h;
    if (lo) lo[e] = l;
  }
}
struct F_k_split_rows {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_split_rows_body(b, g, a...);
  }
};
__global__ void k_split_rows(const double* X, u16* hi, u16* lo, int M, int K, int Kp, int transpose) {
  k_split_rows_body(blockIdx3(), gridDim3(), X, hi, lo, M, K, Kp, transpose);
}
template <int NS>
__device__ __forceinline__ void k_debug_gemm_bf16_body(const uint3 bid_, const uint3 gdim_, const u16* Ah, const u16* Al, const u16* Bh, const u16* Bl,
                                                          float* C, int M, int N, int Kp) {
  using Eng = MmaBF16<64, 128, 2, 2, NS, NS>;
  __shared__ __attribute__((aligned(16))) u16 lds[Eng::LDS_BYTES / 2];
  const int r0 = bid_.y * 64, c0 = bid_.x * 128;
  Eng e;
  e.run([&](int c, int r) -> const u16* { return r0 + r < M ? (c ? Al : Ah) + (int64_t)(r0 + r) * Kp : nullptr; },
        [&](int c, int q) -> const u16* { return c0 + q < N ? (c ? Bl : Bh) + (int64_t)(c0 + q) * Kp : nullptr; },
        Kp, lds);
  e.store([&](int r, int c, float v) {
    if (r0 + r < M && c0 + c < N) C[(int64_t)(r0 + r) * N + c0 + c] = v;
  });
}
template <int NS>
struct F_k_debug_gemm_bf16 {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_debug_gemm_bf16_body<NS>(b, g, a...);
  }
};
template <int NS>
__global__ __launch_bounds__(256) void k_debug_gemm_bf16(const u16* Ah, const u16* Al, const u16* Bh, const u16* Bl,
                                                          float* C, int M, int N, int Kp) {
  k_debug_gemm_bf16_body<NS>(blockIdx3(), gridDim3(), Ah, Al, Bh, Bl, C, M, N, Kp);
}
void launch_debug_gemm_bf16(const double* A, const double* B, float* C, int M, int N, int K, int passes,
                            void* scratch, hipStream_t st) {
  const int Kp = (K + 7) / 8 * 8;
  u16* Ah = (u16*)scratch;
  u16* Al = Ah + (int64_t)M * Kp;
  u16* Bh = Al + (int64_t)M * Kp;
  u16* Bl = Bh + (int64_t)N * Kp;
  afq::glaunch<F_k_split_rows>(k_split_rows, dim3(256), dim3(256), 0, st, A, Ah, Al, M, K, Kp, 0);
  afq::glaunch<F_k_split_rows>(k_split_rows, dim3(256), dim3(256), 0, st, B, Bh, Bl, N, K, Kp, 1);
  dim3 grid(cdivu(N, 128), cdivu(M, 64));
  if (passes == 3)
    afq::glaunch<F_k_debug_gemm_bf16<2>>(k_debug_gemm_bf16<2>, grid, dim3(256), 0, st, Ah, Al, Bh, Bl, C, M, N, Kp);
  else
    afq::glaunch<F_k_debug_gemm_bf16<1>>(k_debug_gemm_bf16<1>, grid, dim3(256), 0, st, Ah, Al, Bh, Bl, C, M, N, Kp);
}

void launch_copy_small(const double* a, double* b, int n, hipStream_t st) {
  afq::glaunch<F_k_copy_calib>(k_copy_calib, dim3(cdivu(n, 256)), dim3(256), 0, st, a, b, (int64_t)n);
}
void launch_copy_calib(const double* a, double* b, int64_t n, hipStream_t st) {
  afq::glaunch<F_k_copy_calib>(k_copy_calib, dim3(2048), dim3(256), 0, st, a, b, n);
}

__device__ __forceinline__ void k_fill_body(const uint3 bid_, const uint3 gdim_, double* p, int64_t n, double v) {
  for (int64_t i = (int64_t)bid_.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gdim_.x * blockDim.x) p[i] = v;
}
struct F_k_fill {
  static constexpr int NT = 1024, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_fill_body(b, g, a...);
  }
};
__global__ void k_fill(double* p, int64_t n, double v) {
  k_fill_body(blockIdx3(), gridDim3(), p, n, v);
}
void launch_fill(double* p, int64_t n, double v, hipStream_t st) {
  if (n <= 0) return;
  afq::glaunch<F_k_fill>(k_fill, dim3((unsigned)std::min<int64_t>(1024, (n + 255) / 256)), dim3(256), 0, st, p, n, v);
}

}  // namespace afq
