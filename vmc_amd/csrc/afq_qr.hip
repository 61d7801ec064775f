// Thin Householder QR of every walker's determinants with Eigen's conventions
// (eigen/Eigen/src/Householder/Householder.h:63-92, eigen/Eigen/src/QR/HouseholderQR.h:267-297);
// psi_d := Q, logO -= log prod diag R (DQMC/DQMCWalker.cpp:295-326).
#include <float.h>

#include "afq_device.hpp"
#include "afq_internal.hpp"

namespace afq {

// One workgroup per walker, its determinants in turn.  Lane c of every wave holds column c (at
// most 64), wave q the rows q, q + WAVES, ..; MR rows a lane, in registers throughout.  Column k
// reaches the other lanes by readlane, so a reflector's products with all columns are lane-local
// sums over a wave's rows, and one exchange of the waves' sums through LDS (two buffers, one
// barrier) is all a step needs: with x the column below the diagonal, c0 its diagonal element and
// s_c = x^* a_c, the column's tail norm is s_k, and beta, tau and den = c0 - beta follow in
// every lane; v = x / den, so v^* a_c = a_kc + conj(1 / den) s_c and a_c -= x (tau v^* a_c / den).
// The columns keep x until all are done and are then scaled to v.  Q = H_0^* .. H_{n-1}^* [I; 0]
// is formed in place, last reflector first: t_c = v^* q_c over the rows below k, row k becomes
// -conj(tau) t_c, q_c -= v conj(tau) t_c, and column k itself turns into e_k - conj(tau) v.
//
// Bound by VALU issue in a serial chain: n steps, each with four lane broadcasts and eight FMAs
// per live row and wave, then one barrier, a square root and three divisions.  A lane that holds
// its column in registers needs neither LDS traffic nor a second barrier; keeping the columns in
// LDS, or in registers with a block-wide reduction for the norm and one for the products, took at
// N = 10 (128 walkers, n = 5) 31 us, now 11; N = 51 (256, n = 13) 140, now 70; N = 100 (1024,
// n = 20) 1454, now 492; N = 300 (256, n = 60) 1840, now 1015, and 27.7 ms, now 16.2, for 4096.
// Masking the rows above the diagonal instead of zeroing them costs 604 us at N = 100.
constexpr int QC = 4;
template <int WAVES, int MR>
__device__ __forceinline__ void k_qr_cols_body(const uint3 bid_, const uint3 gdim_, double* psi, double* logO,
                                               const double* weights, int N, int ndets, int na, int nb, int64_t offb,
                                               int64_t ms, int rhf_walker) {
  __shared__ __attribute__((aligned(16))) cplx part[2][WAVES][64];
  __shared__ __attribute__((aligned(16))) cplx rowk[2][64];
  __shared__ cplx taus[64], rdens[64];
  __shared__ double betas[64];
  const int w = bid_.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (weights[w] == 0.0) return;   // weight zero: never read again before the comb replaces it
  double lf_re = 0.0, lf_im = 0.0;
  for (int d = 0; d < ndets; ++d) {
    const int n = d == 0 ? na : nb;
    cplx* A = reinterpret_cast<cplx*>(psi + 2 * ((int64_t)w * ms + (d == 0 ? 0 : offb)));
    cplx a[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const int i = wave + WAVES * m;
      a[m] = cplx{0.0, 0.0};
      if (i < N && lane < n) a[m] = A[(unsigned)(i * n + lane)];
    }
    // Row k of the columns from k on is R, which nothing reads after its step: it is zeroed as it
    // is taken out, so that the rows above a reflector need no masks.  Rows go in chunks of QC;
    // one that lies above row k (or past N) is passed over.  The bounds are opaque to the
    // compiler, which would keep each chunk's condition in scalar registers otherwise.
    const int nc = (N + WAVES * QC - 1) / (WAVES * QC);
    auto each = [&](int k, int mk, auto f) {
      int ncl = nc;
      asm volatile("" : "+s"(ncl), "+s"(mk));
#pragma unroll
      for (int c = 0; c < MR / QC; ++c) {
        if (c >= ncl || QC * (c + 1) <= mk) continue;
#pragma unroll
        for (int m = QC * c; m < QC * (c + 1); ++m) f(m, readlane_f64(a[m].re, k), readlane_f64(a[m].im, k));
      }
    };
    auto take = [&](int mk, bool mine) {   // a[mk], which becomes 0 where it is mine
      cplx e{0.0, 0.0};
      asm volatile("" : "+s"(mk));
#pragma unroll
      for (int c = 0; c < MR / QC; ++c) {
        if (mk / QC != c) continue;
#pragma unroll
        for (int m = QC * c; m < QC * (c + 1); ++m) {
          const bool at = m == mk;
          e.re = at ? a[m].re : e.re;
          e.im = at ? a[m].im : e.im;
          a[m].re = at && mine ? 0.0 : a[m].re;
          a[m].im = at && mine ? 0.0 : a[m].im;
        }
      }
      return e;
    };
    auto put = [&](int mk, bool mine, cplx e) {
      asm volatile("" : "+s"(mk));
#pragma unroll
      for (int c = 0; c < MR / QC; ++c) {
        if (mk / QC != c) continue;
#pragma unroll
        for (int m = QC * c; m < QC * (c + 1); ++m) {
          const bool at = mine && m == mk;
          a[m].re = at ? e.re : a[m].re;
          a[m].im = at ? e.im : a[m].im;
        }
      }
    };
    // this wave's share of x_k^* a_c over the rows below k
    auto dot = [&](int k, int mk) {
      cplx s{0.0, 0.0}, t{0.0, 0.0};
      each(k, mk, [&](int m, double xr, double xi) {
        s.re += xr * a[m].re;
        t.re += xi * a[m].im;
        s.im += xr * a[m].im;
        t.im -= xi * a[m].re;
      });
      return cadd(s, t);
    };
    // a_c -= x_k g over the same rows
    auto update = [&](int k, int mk, cplx g) {
      each(k, mk, [&](int m, double xr, double xi) {
        a[m].re -= xr * g.re;
        a[m].im -= xr * g.im;
        a[m].re += xi * g.im;
        a[m].im -= xi * g.re;
      });
    };
    auto total = [&](int buf) {
      cplx s = part[buf][0][lane];
#pragma unroll
      for (int q = 1; q < WAVES; ++q) s = cadd(s, part[buf][q][lane]);
      return s;
    };
    for (int k = 0; k < n; ++k) {
      const int buf = k & 1, mk = k / WAVES, wk = k - mk * WAVES;   // row k: slot mk of wave wk
      if (wave == wk) rowk[buf][lane] = take(mk, lane >= k);
      part[buf][wave][lane] = dot(k, mk);
      __syncthreads();
      const cplx s = total(buf), akc = rowk[buf][lane];
      const double tail = readlane_f64(s.re, k);
      const cplx c0{readlane_f64(akc.re, k), readlane_f64(akc.im, k)};
      const bool zero = tail <= DBL_MIN && c0.im * c0.im <= DBL_MIN;
      double beta = c0.re;
      cplx rden{0.0, 0.0}, tau{0.0, 0.0};
      if (!zero) {
        beta = sqrt(c0.re * c0.re + c0.im * c0.im + tail);
        if (c0.re >= 0.0) beta = -beta;
        // 1 / den: beta has the sign opposite to c0.re, so |re| >= |im| (Smith's division)
        const double dr = c0.re - beta, q = c0.im / dr, id = 1.0 / (dr + c0.im * q);
        rden = cplx{id, -q * id};
        const double rb = 1.0 / beta;
        tau = cplx{(beta - c0.re) * rb, c0.im * rb};   // conj((beta - c0) / beta)
      }
      if (tid == 0) {
        taus[k] = tau;
        rdens[k] = rden;
        betas[k] = beta;
      }
      const cplx tmp = cadd(akc, cmul(cplx{rden.re, -rden.im}, s));
      cplx u = cmul(tau, tmp);
      if (lane <= k) u = cplx{0.0, 0.0};
      update(k, mk, cmul(u, rden));
    }
    __syncthreads();   // taus, rdens, betas; and the buffers are free again
    if (wave == 0) {
      // log prod beta over this determinant's reflectors
      const double lb = lane < n ? log(fabs(betas[lane])) : 0.0;
      const double ng = (lane < n && betas[lane] < 0.0) ? 1.0 : 0.0;
      lf_re += wave_sum(lb);
      lf_im += M_PI * wave_sum(ng);
    }
    {
      const cplx rd = rdens[lane < n ? lane : 0];
#pragma unroll
      for (int m = 0; m < MR; ++m) a[m] = cmul(a[m], rd);   // x -> v
    }
    for (int k = n - 1; k >= 0; --k) {
      const int buf = k & 1, mk = k / WAVES, wk = k - mk * WAVES;
      part[buf][wave][lane] = dot(k, mk);
      __syncthreads();
      const cplx tk = taus[k], ct{tk.re, -tk.im};
      const cplx t = cmul(ct, total(buf));
      cplx g = t, r{-t.re, -t.im};          // columns past k
      if (lane == k) {
        g = cplx{1.0 + ct.re, ct.im};       // v - v (1 + conj(tau))
        r = cplx{1.0 - ct.re, -ct.im};
      }
      if (lane < k) g = cplx{0.0, 0.0};
      update(k, mk, g);
      if (wave == wk) put(mk, lane >= k, r);
    }
    // the bounds anew (opaque to the compiler), so that the loads' masks are not kept in scalar
    // registers through the whole factorisation
    int N2 = N, n2 = n;
    asm volatile("" : "+s"(N2), "+s"(n2));
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const int i = wave + WAVES * m;
      if (i < N2 && lane < n2) A[(unsigned)(i * n2 + lane)] = a[m];
    }
    __syncthreads();   // before the next determinant reuses the buffers
  }
  if (tid == 0) {
    const double m = rhf_walker ? 2.0 : 1.0;
    logO[2 * w] -= m * lf_re;
    logO[2 * w + 1] -= m * lf_im;
  }
}
template <int WAVES, int MR>
struct F_k_qr_cols {
  static constexpr int NT = 64 * WAVES, OCC = MR <= 16 ? 4 : 2;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_qr_cols_body<WAVES, MR>(b, g, a...);
  }
};
template <int WAVES, int MR>
__global__ __launch_bounds__(64 * WAVES, MR <= 16 ? 4 : 2) void k_qr_cols(double* psi, double* logO, const double* weights,
                                                                        int N, int ndets, int na, int nb, int64_t offb,
                                                                        int64_t ms, int rhf_walker) {
  k_qr_cols_body<WAVES, MR>(blockIdx3(), gridDim3(), psi, logO, weights, N, ndets, na, nb, offb, ms, rhf_walker);
}

template <int WAVES, int MR>
static void go(const DevState& s, hipStream_t st) {
  afq::glaunch<F_k_qr_cols<WAVES, MR>>((k_qr_cols<WAVES, MR>), dim3(s.W), dim3(64 * WAVES), 0, st, s.psi, s.logO, s.weights, s.N,
                                       s.ndets_prop, s.det_n[0], s.det_n[1], s.det_off[1], s.ms, (int)s.walker_rhf);
}
// A column takes one lane (a context has at most 64 electrons of a spin) and its rows 4 MR registers a lane.  Four waves leave two
// workgroups on a CU up to N = 128; past it eight waves keep MR within the 256 registers that two
// waves a SIMD may use, up to N = 320.  Past that the columns stay in memory (k_qr).
bool launch_qr_cols(const DevState& s, hipStream_t st) {
  if (s.N > 320) return false;
  if (s.N <= 32) go<4, 8>(s, st);
  else if (s.N <= 64) go<4, 16>(s, st);
  else if (s.N <= 96) go<4, 24>(s, st);
  else if (s.N <= 128) go<4, 32>(s, st);
  else if (s.N <= 192) go<8, 24>(s, st);
  else if (s.N <= 256) go<8, 32>(s, st);
  else go<8, 40>(s, st);
  return true;
}

}  // namespace afq
