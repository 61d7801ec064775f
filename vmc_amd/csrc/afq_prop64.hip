// The whole FP64 propagation of a block of one walker's columns in one workgroup:
//   x <- E (sum_{k<=5} V^k / k!) E x,   V = i sqrt(dt) P
// (DQMC/DQMCWalker.cpp:424-431,482-491; with unrestricted integrals each determinant has
// its own E and P, :506-554), the Taylor sum by Horner's rule u <- t0 + (V u) / p, p = 5..1.
//
// The block (8 CT complex columns = 16 CT real ones, all N orbitals) stays in LDS for the
// seven products as u[orbital][re, im interleaved], the B operand of every MFMA.  The
// complex product is the real one with P_im against (u_re, u_im) and P_re against
// (u_im, -u_re): V u = -sqrt(dt) (P_im b1 + P_re b2), b2 being b1's neighbour column with
// the sign of the imaginary lanes flipped.  P is symmetric, so a lane's A element
// P(row, k) is read at [k][row] and the 16 lanes of a row tile read 128 contiguous bytes;
// the A operands go from global memory straight to registers NS - 1 K steps ahead, because
// each wave owns its row tiles (wave, wave + 4, ..) and shares them with no other.  A
// product needs no barrier, one Horner step two.  t0 = E x stays in registers.  Walkers at or
// below the propagation threshold are skipped.
//
// Bound by FP64 MFMA issue: four waves, up to six row tiles each, so that a K step is up to
// 40 independent MFMAs and one wave per SIMD keeps the pipe full.  Before, two one-body and
// five Taylor launches moved every term through HBM, with 64 x 128 tiles and element
// loaders up to 64 electrons: 2.31 ms a step at N = 100, 20+20, 1024 walkers, now 0.41
// (48 TFLOP/s; 7 row tiles on 4 waves leave 7/8 at most); 4.16 -> 2.31 ms (57 TFLOP/s) at
// N = 300, 60+60, 256 walkers; 56 -> 5.6 us at N = 10, 5+5, 128 walkers.
#include <algorithm>
#include <utility>

#include "afq_device.hpp"
#include "afq_internal.hpp"

namespace afq {

static inline unsigned cdivu(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

constexpr int P64_WAVES = 4;
template <int MT, int CT>
struct Prop64Shape {
  static constexpr int NT = 64 * P64_WAVES;
  static constexpr int ROWS = 16 * P64_WAVES * MT;   // orbitals held; N at most this
  static constexpr int LD = 16 * CT;                 // real columns
  static constexpr int NS = MT <= 2 ? 4 : 3;         // A register sets
  static constexpr int OCC = MT == 1 ? 3 : MT == 2 ? 2 : 1;
};

template <int MT, int CT>
__device__ __forceinline__ void k_prop64_body(const uint3 bid_, const uint3 gdim_, const double* P0, const double* P1,
                                              const double* E0, const double* E1, const double* src, double* dst,
                                              const double* weights, int N, int na, int nb, int64_t offb, int64_t wstride,
                                              double sq, int nblk0, int nblk1, int W) {
  using S = Prop64Shape<MT, CT>;
  constexpr int LD = S::LD, NS = S::NS;
  __shared__ __attribute__((aligned(16))) double u[S::ROWS * LD];
  const int nblk = nblk0 + nblk1;
  const TileId tl = tile_id_at(bid_.x, nblk, 1, W, 1);
  const int w = tl.z;
  if (weights[w] <= 1e-8) return;
  const bool second = tl.x >= nblk0;                  // the down spin's own block (unrestricted integrals)
  const int q0 = (second ? tl.x - nblk0 : tl.x) * 8 * CT;
  const int ncol = second ? nb : nblk1 > 0 ? na : na + nb;
  const int lane = threadIdx.x & 63, cl = lane & 15, kh = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int RT = (N + 15) >> 4, nk = (N + 3) >> 2;
  const double* Pre = (second ? P1 : P0) + (int64_t)(2 * w) * N * N;
  const double* Pim = Pre + (int64_t)N * N;
  const double* E = second ? E1 : E0;
  const double* xs = src + (int64_t)w * wstride;
  double* xd = dst + (int64_t)w * wstride;

  int rt[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) rt[m] = wave + P64_WAVES * m;
  // offset of (row, this lane's column of column tile j) in the walker: cb[j] + row rs[j]
  int cb[CT], rs[CT];
  auto col_setup = [&](int qb) {
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int q = qb + 8 * j + (cl >> 1), comp = cl & 1;
      const bool up = !second && q < na;
      cb[j] = up ? 2 * q + comp : (int)(2 * (offb + (second ? q : q - na))) + comp;
      rs[j] = q < ncol ? (up ? 2 * na : 2 * nb) : -1;   // -1: padding column
    }
  };
  col_setup(q0);
  // u offset of (row, real column 16 j + c) less row LD + 16 j, for this lane's rows, whose
  // parity is kh's (they are kh modulo 4).  With an even CT, rows k and k + 1 would start on
  // the same bank; odd rows swap the column tiles 2 i and 2 i + 1 instead.
  const int sw = CT % 2 == 0 ? 16 * (kh & 1) : 0;
  auto at = [&](int j) { return j & 1 ? cl - sw : cl + sw; };
  auto at2 = [&](int j) { return j & 1 ? (cl ^ 1) - sw : (cl ^ 1) + sw; };

  f64x4 T[MT][CT], acc[MT][CT];
  auto put = [&](const f64x4 (&v)[MT][CT]) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (rt[m] >= RT) continue;   // wave-uniform
#pragma unroll
      for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * rt[m] + kh + 4 * r;
          u[row * LD + 16 * j + at(j)] = row < N ? v[m][j][r] : 0.0;   // orbital pads stay zero
        }
    }
  };
  // A operands of K step s (k = 4 s + lane / 16) of the real E and of P; rows and k past N
  // read a valid neighbour: those k meet zero rows of u, those rows are never stored
  int er[MT], pr[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    pr[m] = min(16 * rt[m] + cl, N - 1);
    er[m] = pr[m] * N;
  }
  double A0[NS][MT], A1[NS][MT];
  auto loadE = [&](int s, int set) {
    const int k = min(4 * s + kh, N - 1);
#pragma unroll
    for (int m = 0; m < MT; ++m) A0[set][m] = E[er[m] + k];
  };
  auto loadP = [&](int s, int set) {
    const int k = min(4 * s + kh, N - 1) * N;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      A0[set][m] = Pim[k + pr[m]];
      A1[set][m] = Pre[k + pr[m]];
    }
  };
  auto stepE = [&](int s, int set) {
    const int k = 4 * s + kh;
    double b[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) b[j] = u[k * LD + 16 * j + at(j)];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (rt[m] >= RT) continue;
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[m][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(A0[set][m], b[j], acc[m][j], 0, 0, 0);
    }
  };
  const unsigned flip = (cl & 1) ? 0x80000000u : 0u;
  auto stepP = [&](int s, int set) {
    const int k = 4 * s + kh;
    double b1[CT], b2[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) b1[j] = u[k * LD + 16 * j + at(j)];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const double v = u[k * LD + 16 * j + at2(j)];
      b2[j] = __hiloint2double(__double2hiint(v) ^ flip, __double2loint(v));
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (rt[m] >= RT) continue;
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[m][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(A0[set][m], b1[j], acc[m][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[m][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(A1[set][m], b2[j], acc[m][j], 0, 0, 0);
    }
  };
  auto pre = [&](auto load) {
#pragma unroll
    for (int i = 0; i + 1 < NS; ++i) load(i, i);
  };
  // the nk K steps of one product, whose first NS - 1 are already requested
  auto product = [&](auto load, auto step) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[m][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    int s = 0;
    for (; s + NS <= nk; s += NS) {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        load(s + i + NS - 1, (i + NS - 1) % NS);
        step(s + i, i);
      }
    }
#pragma unroll
    for (int i = 0; i + 1 < NS; ++i)
      if (s + i < nk) step(s + i, i);
  };

  pre(loadE);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * rt[m] + kh + 4 * r;
        T[m][j][r] = row < N && rs[j] >= 0 ? xs[cb[j] + (int64_t)row * rs[j]] : 0.0;
      }
  put(T);
  __syncthreads();
  product(loadE, stepE);   // t0 = E x
  pre(loadP);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < CT; ++j) T[m][j] = acc[m][j];
  __syncthreads();
  put(acc);
  __syncthreads();
  for (int p = 5; p >= 1; --p) {
    product(loadP, stepP);
    if (p > 1) pre(loadP);
    else pre(loadE);
    const double f = -sq / (double)p;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][j][r] = T[m][j][r] + f * acc[m][j][r];
    __syncthreads();
    put(acc);
    __syncthreads();
  }
  product(loadE, stepE);
  // the column offsets again from scratch (opaque to the compiler), so that the prologue's
  // addresses are not kept live through the whole kernel
  int q0o = q0;
  asm volatile("" : "+v"(q0o));
  col_setup(q0o);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * rt[m] + kh + 4 * r;
        if (row < N && rs[j] >= 0) xd[cb[j] + (int64_t)row * rs[j]] = acc[m][j][r];
      }
}
template <int MT, int CT>
struct F_k_prop64 {
  static constexpr int NT = Prop64Shape<MT, CT>::NT, OCC = Prop64Shape<MT, CT>::OCC;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_prop64_body<MT, CT>(b, g, a...);
  }
};
template <int MT, int CT>
__global__ __launch_bounds__(64 * P64_WAVES, MT == 1 ? 3 : MT == 2 ? 2 : 1) void k_prop64(const double* P0, const double* P1, const double* E0,
                                                                    const double* E1, const double* src, double* dst,
                                                                    const double* weights, int N, int na, int nb,
                                                                    int64_t offb, int64_t wstride, double sq, int nblk0,
                                                                    int nblk1, int W) {
  k_prop64_body<MT, CT>(blockIdx3(), gridDim3(), P0, P1, E0, E1, src, dst, weights, N, na, nb, offb, wstride, sq, nblk0,
                        nblk1, W);
}

bool prop64_fits(const DevState& s) { return s.N <= 384; }

template <int MT, int CT>
static void go(const DevState& s, double* dst, int nblk0, int nblk1, hipStream_t st) {
  using S = Prop64Shape<MT, CT>;
  if constexpr (S::ROWS * S::LD * 8 <= 160 * 1024)
    afq::glaunch<F_k_prop64<MT, CT>>((k_prop64<MT, CT>), dim3((unsigned)((nblk0 + nblk1) * s.W)), dim3(S::NT), 0, st, s.P,
                                     s.uints ? s.P2 : s.P, s.E, s.uints ? s.E2 : s.E, s.psi, dst, s.weights, s.N, s.det_n[0],
                                     s.ndets_prop > 1 ? s.det_n[1] : 0, s.det_off[1], 2 * s.ms, sqrt(s.dt), nblk0, nblk1,
                                     s.W);
}
template <int MT>
static void go_ct(const DevState& s, int ct, double* dst, int nblk0, int nblk1, hipStream_t st) {
  switch (ct) {
    case 1: go<MT, 1>(s, dst, nblk0, nblk1, st); break;
    case 2: go<MT, 2>(s, dst, nblk0, nblk1, st); break;
    case 3: go<MT, 3>(s, dst, nblk0, nblk1, st); break;
    case 4: go<MT, 4>(s, dst, nblk0, nblk1, st); break;
    default: go<MT, 5>(s, dst, nblk0, nblk1, st); break;
  }
}
void launch_prop64(const DevState& s, double* dst, hipStream_t st) {
  const int na = s.det_n[0], nb = s.ndets_prop > 1 ? s.det_n[1] : 0;
  // column tiles of 8 complex columns of the (one or two) groups that share a P
  const int t0 = (int)cdivu(s.uints ? na : na + nb, 8), t1 = s.uints ? (int)cdivu(nb, 8) : 0;
  // A workgroup's time is its column tiles' MFMAs, and workgroups that share a CU share its
  // MFMA pipes, so a launch takes (blocks per CU, rounded up) x ct; among equals the widest
  // block, which reads P least often.  N = 300, 15 tiles, 256 walkers: ct 3 (5 x 3) 2.31 ms,
  // 4 (4 x 4) 2.50, 2 (8 x 2) 2.65; 64 walkers: ct 4 (1 x 4) 0.64 ms, 3 (2 x 3) 0.91; 16
  // walkers: ct 1 (1 x 1) 0.23 ms, 4 (1 x 4) 0.61.  N = 100, 5 tiles, 1024 walkers: ct 5
  // 0.41 ms, 3 0.50, 2 0.53; 64 walkers: ct 2 0.057 ms, 5 0.115.
  const int ctmax = std::min(s.N <= 256 ? 5 : s.N <= 320 ? 4 : 3, std::max(t0, t1));   // what the LDS holds
  int ct = 1, nblk0 = t0, nblk1 = t1;
  int64_t best = INT64_MAX;
  for (int c = ctmax; c >= 1; --c) {
    const int n0 = (int)cdivu(t0, c), n1 = (int)cdivu(t1, c);
    const int64_t cost = (int64_t)cdivu((int64_t)(n0 + n1) * s.W, 256) * c;
    if (cost < best) {
      best = cost;
      ct = c;
      nblk0 = n0;
      nblk1 = n1;
    }
  }
  switch ((int)cdivu(s.N, 64)) {
    case 1: go_ct<1>(s, ct, dst, nblk0, nblk1, st); break;
    case 2: go_ct<2>(s, ct, dst, nblk0, nblk1, st); break;
    case 3: go_ct<3>(s, ct, dst, nblk0, nblk1, st); break;
    case 4: go_ct<4>(s, ct, dst, nblk0, nblk1, st); break;
    case 5: go_ct<5>(s, ct, dst, nblk0, nblk1, st); break;
    default: go_ct<6>(s, ct, dst, nblk0, nblk1, st); break;
  }
}

}  // namespace afq
