// FP64 VHS P[(w,c), t] = sum_g field[w][g][c] Lp[g][t] (DQMC/DQMCWalker.cpp:406-421), t running
// over the packed lower triangle; with unrestricted integrals also the down-spin VHS from the
// down-spin vectors (propagatePhaselessU, DQMC/DQMCWalker.cpp:525-530).
#include <algorithm>

#include "afq_gemm64.hpp"
#include "afq_internal.hpp"

namespace afq {

static inline unsigned cdivu(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

// A wave takes 16 A walkers (their real and imaginary rows are two row tiles, fed by one 16-byte
// load of a field) times 2 B blocks of 4 x 4 matrix elements (adjacent pairs of a row are two
// column tiles, likewise fed by one 16-byte load; the packed elements of a row are contiguous); a
// workgroup 2 x 2 waves.  Operands go from memory straight to registers, NS - 1 K steps ahead;
// waves of a workgroup share them through the first-level cache.  Lp holds a double past its end.
//
// Bound by FP64 MFMA issue and by the stores of the full N x N matrices that the propagation
// reads.  With columns in packed order the upper triangle's elements went out one 8-byte store
// to a line, 100 of 275 us at N = 100, G = 400, 1024 walkers; in 4 x 4 blocks they go in runs
// of 32 bytes (16 x 16 or 8 x 8 blocks would pad the triangle by 15 % there, these by 3 %).
// Through LDS with 128 x 128 tiles this took 286 us there, now 190 (44 TFLOP/s with 164 MB
// written); N = 300, G = 1200, 256 walkers 1280, now 978 (57 TFLOP/s); N = 51, G = 205, 256
// walkers, both spins 104, now 24.
template <int A, int B>
struct VhsShape {
  static constexpr int NS = 3, BM = 32 * A, BN = 64 * B;
};
template <int A, int B>
__device__ __forceinline__ void k_vhs64_body(const uint3 bid_, const uint3 gdim_, const double* fields, const double* Lp0,
                                             const double* Lp1, double* P0, double* P1, const double* weights, int G, int W,
                                             int T, int N, int ref_compat, int gridx, int gridy, int gridz) {
  using S = VhsShape<A, B>;
  constexpr int NS = S::NS;
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, gridz, 1);
  const int lane = threadIdx.x & 63, cl = lane & 15, kh = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w0 = tl.y * S::BM + 16 * A * (wave >> 1), t0 = tl.x * S::BN + 32 * B * (wave & 1);
  const int nb4 = (N + 3) >> 2, nblk = nb4 * (nb4 + 1) / 2;
  if (w0 >= W || t0 >= 16 * nblk) return;
  // a tile whose walkers are all dead is skipped
  if (__ballot(lane < 16 * A && w0 + lane < W && weights[min(w0 + lane, W - 1)] > 1e-8) == 0) return;
  // columns go in 4 x 4 blocks of the lower triangle, block (i, j) at i (i + 1) / 2 + j; this
  // lane's pair (row, col), (row, col + 1) of the two blocks from column t on
  auto column = [&](int t, int& row, int& col) {
    const int b = (t >> 4) + ((cl >> 1) & 1);
    int i = (int)((sqrtf(8.0f * (float)b + 1.0f) - 1.0f) * 0.5f);
    if ((i + 1) * (i + 2) / 2 <= b) ++i;
    if (i * (i + 1) / 2 > b) --i;
    row = 4 * i + (cl >> 2);
    col = 4 * (b - i * (i + 1) / 2) + 2 * (cl & 1);
  };
  const double* Lp = tl.z == 0 ? Lp0 : Lp1;
  double* P = tl.z == 0 ? P0 : P1;
  // walkers and columns past the data read a valid one
  const double* pa[A];
  unsigned tc[B];
#pragma unroll
  for (int i = 0; i < A; ++i) pa[i] = fields + (int64_t)min(w0 + 16 * i + cl, W - 1) * 2 * G;
#pragma unroll
  for (int j = 0; j < B; ++j) {
    int r, c;
    column(t0 + 32 * j, r, c);
    tc[j] = min(r * (r + 1) / 2 + c, T - 1);
  }
  const int nk = (G + 3) >> 2;
  f64x2 a[NS][A], b[NS][B];
  auto load = [&](int s, int set) {
    s = min(s, nk - 1);
    const int kc = min(kh, G - 1 - 4 * s);
#pragma unroll
    for (int i = 0; i < A; ++i) a[set][i] = *reinterpret_cast<const f64x2*>(pa[i] + 2 * (4 * s + kc));
    const double* base = Lp + (int64_t)4 * s * T;
#pragma unroll
    for (int j = 0; j < B; ++j) b[set][j] = load2(base + (unsigned)(kc * T + tc[j]));
  };
  f64x4 acc[A][2][B][2];
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j)
#pragma unroll
      for (int c = 0; c < 2; ++c) acc[i][c][j][0] = acc[i][c][j][1] = f64x4{0.0, 0.0, 0.0, 0.0};
  auto step = [&](int set) {
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
      for (int j = 0; j < B; ++j) {
        acc[i][0][j][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[set][i].x, b[set][j].x, acc[i][0][j][0], 0, 0, 0);
        acc[i][0][j][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[set][i].x, b[set][j].y, acc[i][0][j][1], 0, 0, 0);
        acc[i][1][j][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[set][i].y, b[set][j].x, acc[i][1][j][0], 0, 0, 0);
        acc[i][1][j][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[set][i].y, b[set][j].y, acc[i][1][j][1], 0, 0, 0);
      }
  };
#pragma unroll
  for (int i = 0; i + 1 < NS; ++i) load(i, i);
  int s = 0;
  for (; s + NS < nk; s += NS) {
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      load(s + i + NS - 1, (i + NS - 1) % NS);
      step(i);
    }
  }
  // the last one to NS steps (NS - 1 of them requested); k past G add nothing
  if (s + NS - 1 < nk) load(s + NS - 1, NS - 1);
#pragma unroll
  for (int i = 0; i < NS; ++i)
    if (s + i < nk) {
      if (4 * (s + i) + kh >= G) {
#pragma unroll
        for (int q = 0; q < A; ++q) a[i][q] = f64x2{0.0, 0.0};
#pragma unroll
        for (int q = 0; q < B; ++q) b[i][q] = f64x2{0.0, 0.0};
      }
      step(i);
    }
  // both triangles of the N x N matrix
#pragma unroll
  for (int q = 0; q < B; ++q) {
    int i, j;
    column(t0 + 32 * q, i, j);
    if (i >= N || j > i) continue;
#pragma unroll
    for (int p = 0; p < A; ++p)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int w = w0 + 16 * p + kh + 4 * r;
        if (w >= W) continue;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          f64x2 x{acc[p][c][q][0][r], acc[p][c][q][1][r]};
          if (ref_compat) x = f64x2{(double)(float)x.x, (double)(float)x.y};
          double* Pq = P + (int64_t)(2 * w + c) * N * N;
          Pq[j * N + i] = x.x;
          if (j < i) {
            *reinterpret_cast<f64x2u*>(Pq + i * N + j) = f64x2u{x.x, x.y};
            Pq[(j + 1) * N + i] = x.y;
          }
        }
      }
  }
}
template <int A, int B>
struct F_k_vhs64 {
  static constexpr int NT = 256, OCC = A * B == 4 ? 2 : 3;
  static constexpr bool HAS_OCC = true;
  template <class... X>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, X... x) const {
    k_vhs64_body<A, B>(b, g, x...);
  }
};
template <int A, int B>
__global__ __launch_bounds__(256, A * B == 4 ? 2 : 3) void k_vhs64(const double* fields, const double* Lp0, const double* Lp1,
                                                                   double* P0, double* P1, const double* weights, int G, int W,
                                                                   int T, int N, int ref_compat, int gridx, int gridy,
                                                                   int gridz) {
  k_vhs64_body<A, B>(blockIdx3(), gridDim3(), fields, Lp0, Lp1, P0, P1, weights, G, W, T, N, ref_compat, gridx, gridy, gridz);
}

template <class S>
static dim3 tiles(const DevState& s) {
  const int64_t nb4 = (s.N + 3) / 4;
  return dim3(cdivu(8 * nb4 * (nb4 + 1), S::BN), cdivu(s.W, S::BM), s.uints ? 2 : 1);
}
template <class S>
static int64_t workgroups(const DevState& s) {
  const dim3 g = tiles<S>(s);
  return (int64_t)g.x * g.y * g.z;
}
template <int A, int B>
static void go(const DevState& s, hipStream_t st) {
  using S = VhsShape<A, B>;
  const dim3 g = tiles<S>(s);
  afq::glaunch<F_k_vhs64<A, B>>((k_vhs64<A, B>), dim3(g.x * g.y * g.z), dim3(256), 0, st, s.fields, s.Lp, s.Lp2, s.P, s.P2,
                                s.weights, s.G, s.W, (int)s.T, s.N, (int)s.ref_compat, (int)g.x, (int)g.y, (int)g.z);
}
// The larger tile needs fewer loads a product (the first-level cache feeds 64 bytes a clock), the
// smaller one more workgroups: one round of 256 workgroups takes, at G = 400, about 60, 33 and
// 20 us with <2, 2>, <2, 1> and <1, 1>, and the tile with the least rounds times that is taken:
//   N = 100, G = 400:  128 walkers 60, 35, 41 us;  256: 64, 65, 62;  512: 119, 103, 126;
//                      1024: 190, 212, 252
//   N = 300, G = 1200: 16 walkers 288, 171, 142 us;  256: 978, 1259, 1575
//   N = 10, G = 40, 128 walkers: 10, 7, 5 us
// In a grouped launch the other systems fill the chip, and <2, 2> is best whatever the size: 640,
// 746 and 863 us for 24 systems of N = 20 .. 120, 256 walkers each.
void launch_vhs(const DevState& s, hipStream_t st) {
  auto cost = [&](auto shape, int unit) {
    using S = decltype(shape);
    return (int64_t)cdivu(workgroups<S>(s), 256) * unit;
  };
  const int64_t c22 = cost(VhsShape<2, 2>{}, 60), c21 = cost(VhsShape<2, 1>{}, 33), c11 = cost(VhsShape<1, 1>{}, 20);
  if (g_recorder || c22 <= std::min(c21, c11)) go<2, 2>(s, st);
  else if (c21 <= c11) go<2, 1>(s, st);
  else go<1, 1>(s, st);
}

}  // namespace afq
