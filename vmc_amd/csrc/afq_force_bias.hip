// FP64 force bias fb[w][g] = alpha sum_k theta[w][k] R[g][k] over the walkers of nonzero
// weight (DQMC/RHF.cpp:54-61, DQMC/UHF.cpp:45-53), k running over all slots' (orbital,
// electron) pairs.  A walker of weight zero is neither propagated nor measured
// (DQMC/MixedEstimator.cpp:461-468,531) and the comb replaces it, so its force bias is
// never read.  (A walker below the propagation threshold 1e-8 but nonzero is still
// measured, and E_J needs its force bias.)  The grid covers every walker; tiles past the
// live count exit.
#include <algorithm>
#include <cmath>
#include <vector>

#include "afq_gemm64.hpp"
#include "afq_internal.hpp"

namespace afq {

static inline unsigned cdivu(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

// BM real rows (BM / 2 walkers) x BN vectors.  k runs in units of ku, summed in chunks of s units
// each and then over the chunks: an order that only the system decides (fb_order), so that a
// walker's force bias is the same to the last bit in any company.  Workgroup z takes units
// [z m, (z + 1) m).  It writes every unit's sum to part[unit][row][g], or, with whole (m then a
// multiple of s), adds up the chunks itself and writes those; k_fb_reduce does the rest.  With one
// part in all (np) it writes the result.
template <int BM, int BN, int WAVES_M, int WAVES_N>
__device__ __forceinline__ void k_fb64_body(const uint3 bid_, const uint3 gdim_, const double* R, const double* th, double* fb,
                                            double* part, const int* live, const int* nlive, int G, int W, int64_t Ktot,
                                            int ku, int s, int m, int whole, int np, double alpha, int gridx, int gridy,
                                            int gridz) {
  constexpr int NT = 64 * WAVES_M * WAVES_N;
  using SA = StageC<BM, NT>;
  using SB = StageK<BN, NT>;
  using Eng = Gemm64<SA, SB, BM, BN, WAVES_M, WAVES_N>;
  __shared__ __attribute__((aligned(16))) double lds[Eng::LDS_DOUBLES];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, gridz, 8);
  const int row0 = tl.y * BM, g0 = tl.x * BN, nrow = 2 * *nlive;
  if (row0 >= nrow) return;
  SA sa;
  SB sb;
  sa.init([&](int l) -> const double* {
    const int q = row0 / 2 + l;
    return 2 * q < nrow ? th + (int64_t)live[q] * 2 * Ktot : nullptr;
  });
  sb.init([&](int r) -> const double* { return g0 + r < G ? R + (int64_t)(g0 + r) * Ktot : nullptr; });
  Eng e;
  const int k0 = tl.z * m * ku, kend = (int)min((int64_t)k0 + m * ku, Ktot);
  f64x4 sum[Eng::TM][Eng::TN];
  int left = 0;   // units still to come in this part
  int p = tl.z * (whole ? m / s : m), k = k0;
  e.run(sa, sb, k0, kend, lds, ku, [&](const f64x4 (&acc)[Eng::TM][Eng::TN]) {
    if (left == 0) {
      left = whole ? s : 1;
#pragma unroll
      for (int i = 0; i < Eng::TM; ++i)
#pragma unroll
        for (int j = 0; j < Eng::TN; ++j) sum[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    }
#pragma unroll
    for (int i = 0; i < Eng::TM; ++i)
#pragma unroll
      for (int j = 0; j < Eng::TN; ++j) sum[i][j] += acc[i][j];
    k += ku;
    if ((--left > 0 && k < kend) || np == 1) return;
    // (opaque to the compiler, so that the addresses are not kept in registers through the K loop)
    int ld = G, r0 = row0;
    asm volatile("" : "+s"(ld), "+s"(r0));
    double* out = part + (int64_t)p++ * 2 * W * ld;
    e.store(sum, [&](int r, int c, double v) {
      if (r0 + r < nrow && g0 + c < ld) out[(int64_t)(r0 + r) * ld + g0 + c] = v;
    });
  });
  if (np == 1)
    e.store(sum, [&](int r, int c, double v) {
      const int q = row0 + r, g = g0 + c;
      if (q < nrow && g < G) fb[(int64_t)live[q >> 1] * 2 * G + 2 * g + (q & 1)] = alpha * v;
    });
}
constexpr int fb_occ(int bm) { return bm == 32 ? 5 : 4; }   // workgroups on a CU that its LDS allows
template <int BM, int BN, int WAVES_M, int WAVES_N>
struct F_k_fb64 {
  static constexpr int NT = 64 * WAVES_M * WAVES_N, OCC = fb_occ(BM);
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_fb64_body<BM, BN, WAVES_M, WAVES_N>(b, g, a...);
  }
};
template <int BM, int BN, int WAVES_M, int WAVES_N>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, fb_occ(BM)) void k_fb64(const double* R, const double* th, double* fb, double* part,
                                                                    const int* live, const int* nlive, int G, int W,
                                                                    int64_t Ktot, int ku, int s, int m, int whole, int np,
                                                                    double alpha, int gridx, int gridy, int gridz) {
  k_fb64_body<BM, BN, WAVES_M, WAVES_N>(blockIdx3(), gridDim3(), R, th, fb, part, live, nlive, G, W, Ktot, ku, s, m, whole, np,
                                        alpha, gridx, gridy, gridz);
}

// fb of the live walkers from the np parts: sums of s parts in order, added in order
__device__ __forceinline__ void k_fb_reduce_body(const uint3 bid_, const uint3 gdim_, const double* __restrict__ part,
                                                 double* __restrict__ fb, const int* live, const int* nlive, int G, int W,
                                                 double alpha, int np, int s) {
  const int64_t i = (int64_t)bid_.x * blockDim.x + threadIdx.x;
  const int l = (int)(i / G), g = (int)(i - (int64_t)l * G);
  if (l >= *nlive) return;
  const double* p = part + (int64_t)(2 * l) * G + g;
  double re = 0.0, im = 0.0;
  for (int c = 0; c < np; c += s) {
    double cr = 0.0, ci = 0.0;
    for (int z = c; z < min(c + s, np); ++z, p += (int64_t)2 * W * G) {
      cr += p[0];
      ci += p[G];
    }
    re += cr;
    im += ci;
  }
  double* o = fb + (int64_t)live[l] * 2 * G + 2 * g;
  o[0] = alpha * re;
  o[1] = alpha * im;
}
struct F_k_fb_reduce {
  static constexpr int NT = 256, OCC = 1;
  static constexpr bool HAS_OCC = false;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_fb_reduce_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256) void k_fb_reduce(const double* __restrict__ part, double* __restrict__ fb, const int* live,
                                                   const int* nlive, int G, int W, double alpha, int np, int s) {
  k_fb_reduce_body(blockIdx3(), gridDim3(), part, fb, live, nlive, G, W, alpha, np, s);
}

// Bound by FP64 MFMA issue.  K is long (Ktot = N (na + nb), 36,000 at N = 300, 60+60) and
// the output small (2W x G), so without a split of K a few tens of workgroups walk it
// serially: at N = 300, G = 1200, 256 walkers 40 workgroups took 12.5 ms (3.5 TFLOP/s); with
// K split it takes 0.87 ms (51 TFLOP/s) with the sum of the parts.
// 64 x 64 tiles leave room for four workgroups on a CU, whose waves cover each other's
// barriers: 128 x 64 and 128 x 128 tiles took 0.82 and 1.02 ms there (0.080, 0.081, 0.095 ms
// at N = 100, G = 400, 512 walkers).  A grid of at most 64 such tiles gains from 32 x 64
// ones: 11 against 15 us for 16 determinants at N = 100, G = 400 (7 tiles), 15.0 against
// 17.4 us at N = 51, G = 205, 256 walkers (32 tiles); at 112 tiles (N = 100, 512 walkers)
// the 64 x 64 tile is ahead, 80 against 95 us.
//
// The order of a sum is the one with the least time over populations of 16 to 4096 walkers, each
// against the best order for it: units of at least 96 (so that a small population fills the chip), at
// most 48 and no more than the larger borrowed workspace of a context holds, in chunks of which there
// are no more than the smaller one (Sg) holds, which is all that a temporary population has.  Against
// an order chosen for each population: 158 us both at N = 100, G = 400, 1024 walkers, 89 and 87 at 512;
// 0.81 and 0.89 ms at N = 300, 256 walkers, 3.26 and 3.20 at 1024; 80 and 93 us at N = 80, G = 333, 700
// walkers; 137 and 172 at N = 156, 57 closed shells, G = 669, 255 walkers.  Choosing it takes the host 0.3
// ms at N = 100 and 1.1 at most, once a context.
// The time of an order: the fewest rounds of resident workgroups times their K (and 64 for the
// prologue and epilogue), plus the parts' way through memory (W G of them written and read take as
// long as 4e-5 of K, 8e-5 with the smaller tile, whose workgroups take half as long for the same K).
static FbSplit fb_split(FbOrder o, int W, int G, int64_t Ktot, int64_t ws_doubles) {
  FbSplit p;
  p.small = (int64_t)cdivu(G, 64) * cdivu(2 * (int64_t)W, 64) <= 64;
  const int slots = p.small ? 1280 : 1024;   // resident workgroups: LDS allows 5 and 4 on a CU
  const int64_t tiles = (int64_t)cdivu(G, 64) * cdivu(2 * (int64_t)W, p.small ? 32 : 64);
  const int nu = (int)cdivu(Ktot, o.ku);
  p.cost = 1e300;
  for (const bool whole : {false, true}) {
    const int st = whole ? o.s : 1, np = (int)cdivu(nu, st);
    if (np > 1 && (int64_t)np * 2 * W * G > ws_doubles) continue;
    const double through = np > 1 ? (p.small ? 8e-5 : 4e-5) * np * W * G : 0.0;
    for (int q = np > 1 ? 1 : np, last = 0; q <= np; ++q) {   // parts a workgroup
      const int z = (int)cdivu(np, q);
      if (z == last) continue;
      last = z;
      const double cost = (double)((tiles * z + slots - 1) / slots) * (double)(std::min((int64_t)q * st * o.ku, Ktot) + 64) + through;
      if (cost < p.cost) {
        p.cost = cost;
        p.m = q * st;
        p.nz = z;
        p.np = np;
        p.whole = whole;
      }
    }
  }
  if (p.small) p.cost *= 0.5;
  return p;
}
FbOrder fb_order(int G, int64_t Ktot, int nslots) {
  const int64_t in_sg = (int64_t)nslots * GN_MAX * GN_MAX / G, in_ws = std::max(in_sg, Ktot / G);   // parts a workspace holds
  const int most = (int)std::max<int64_t>(1, std::min<int64_t>({Ktot / 96, in_ws, 48}));
  constexpr int NW = 17;
  struct Try { FbOrder o; double t[NW]; };
  std::vector<Try> tries;
  double least[NW];
  std::fill(least, least + NW, 1e300);
  for (int nu = std::max(1, most / 3), ku = 0; nu <= most; ++nu) {
    const int k = (int)cdivu(cdivu(Ktot, nu), G64_BK) * G64_BK, n = (int)cdivu(Ktot, k);
    if (k == ku) continue;
    ku = k;
    for (int b = 1, last = 0; b <= std::min<int64_t>({12, std::max<int64_t>(1, in_sg), n}); ++b) {
      Try y{{k, (int)cdivu(n, b)}, {}};
      if (y.o.s == last) continue;
      last = y.o.s;
      for (int i = 0; i < NW; ++i) {
        const int W = (int)(16.0 * std::exp2(0.5 * i));
        y.t[i] = fb_split(y.o, W, G, Ktot, in_ws * 2 * W * G).cost;
        least[i] = std::min(least[i], y.t[i]);
      }
      tries.push_back(y);
    }
  }
  FbOrder best;
  double lost = 1e300;
  for (const Try& y : tries) {
    double t = 0.0;
    for (int i = 0; i < NW; ++i) t += y.t[i] / least[i];
    if (t < lost) {
      lost = t;
      best = y.o;
    }
  }
  return best;
}

void launch_force_bias(const DevState& s, hipStream_t st) {
  launch_live_list(s, st);
  const FbSplit p = fb_split(s.fbo, s.W, s.G, s.Ktot, s.fbw_doubles);
  const double alpha = (double)s.slot[0].mult;
  const int gx = (int)cdivu(s.G, 64), gy = (int)cdivu(2 * (int64_t)s.W, p.small ? 32 : 64);
  if (p.small)
    afq::glaunch<F_k_fb64<32, 64, 1, 4>>((k_fb64<32, 64, 1, 4>), dim3(gx * gy * p.nz), dim3(256), 0, st, s.R, s.theta, s.fb,
                                         s.fbw, s.live, s.nlive, s.G, s.W, s.Ktot, s.fbo.ku, s.fbo.s, p.m, (int)p.whole, p.np, alpha,
                                         gx, gy, p.nz);
  else
    afq::glaunch<F_k_fb64<64, 64, 2, 2>>((k_fb64<64, 64, 2, 2>), dim3(gx * gy * p.nz), dim3(256), 0, st, s.R, s.theta, s.fb,
                                         s.fbw, s.live, s.nlive, s.G, s.W, s.Ktot, s.fbo.ku, s.fbo.s, p.m, (int)p.whole, p.np, alpha,
                                         gx, gy, p.nz);
  if (p.np > 1)
    afq::glaunch<F_k_fb_reduce>(k_fb_reduce, dim3(cdivu((int64_t)s.W * s.G, 256)), dim3(256), 0, st, s.fbw, s.fb, s.live,
                                s.nlive, s.G, s.W, alpha, p.np, p.whole ? 1 : s.fbo.s);
}

}  // namespace afq
