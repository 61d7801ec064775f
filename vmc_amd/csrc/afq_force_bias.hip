// FP64 force bias fb[w][g] = alpha sum_k theta[w][k] R[g][k] over the walkers of nonzero
// weight (DQMC/RHF.cpp:54-61, DQMC/UHF.cpp:45-53), k running over all slots' (orbital,
// electron) pairs.  A walker of weight zero is neither propagated nor measured
// (DQMC/MixedEstimator.cpp:461-468,531) and the comb replaces it, so its force bias is
// never read.  (A walker below the propagation threshold 1e-8 but nonzero is still
// measured, and E_J needs its force bias.)  The grid covers every walker; tiles past the
// live count exit.
#include <algorithm>

#include "afq_gemm64.hpp"
#include "afq_internal.hpp"

namespace afq {

static inline unsigned cdivu(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

// BM real rows (BM / 2 walkers) x BN vectors; with nz > 1 workgroup z sums k in
// [z kchunk, (z + 1) kchunk) into part[z][row][g], which k_fb_reduce adds up in order.
template <int BM, int BN, int WAVES_M, int WAVES_N>
__device__ __forceinline__ void k_fb64_body(const uint3 bid_, const uint3 gdim_, const double* R, const double* th, double* fb,
                                            double* part, const int* live, const int* nlive, int G, int W, int64_t Ktot,
                                            int kchunk, double alpha, int gridx, int gridy, int nz) {
  constexpr int NT = 64 * WAVES_M * WAVES_N;
  using SA = StageC<BM, NT>;
  using SB = StageK<BN, NT>;
  using Eng = Gemm64<SA, SB, BM, BN, WAVES_M, WAVES_N>;
  __shared__ __attribute__((aligned(16))) double lds[Eng::LDS_DOUBLES];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, nz, 8);
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
  const int k0 = tl.z * kchunk;
  e.run(sa, sb, k0, (int)min((int64_t)k0 + kchunk, Ktot), lds);
  double* out = part + (int64_t)tl.z * 2 * W * G;
  e.store([&](int r, int c, double v) {
    const int q = row0 + r, g = g0 + c;
    if (q >= nrow || g >= G) return;
    if (nz > 1) out[(int64_t)q * G + g] = v;
    else fb[(int64_t)live[q >> 1] * 2 * G + 2 * g + (q & 1)] = alpha * v;
  });
}
template <int BM, int BN, int WAVES_M, int WAVES_N>
struct F_k_fb64 {
  static constexpr int NT = 64 * WAVES_M * WAVES_N, OCC = 2;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_fb64_body<BM, BN, WAVES_M, WAVES_N>(b, g, a...);
  }
};
template <int BM, int BN, int WAVES_M, int WAVES_N>
__global__ __launch_bounds__(64 * WAVES_M * WAVES_N, 2) void k_fb64(const double* R, const double* th, double* fb, double* part,
                                                                    const int* live, const int* nlive, int G, int W,
                                                                    int64_t Ktot, int kchunk, double alpha, int gridx,
                                                                    int gridy, int nz) {
  k_fb64_body<BM, BN, WAVES_M, WAVES_N>(blockIdx3(), gridDim3(), R, th, fb, part, live, nlive, G, W, Ktot, kchunk, alpha, gridx,
                                        gridy, nz);
}

// fb of the live walkers from the nz partial sums, added in order of z
__device__ __forceinline__ void k_fb_reduce_body(const uint3 bid_, const uint3 gdim_, const double* __restrict__ part,
                                                 double* __restrict__ fb, const int* live, const int* nlive, int G, int W,
                                                 double alpha, int nz) {
  const int64_t i = (int64_t)bid_.x * blockDim.x + threadIdx.x;
  const int l = (int)(i / G), g = (int)(i - (int64_t)l * G);
  if (l >= *nlive) return;
  const double* p = part + (int64_t)(2 * l) * G + g;
  double re = 0.0, im = 0.0;
  for (int z = 0; z < nz; ++z, p += (int64_t)2 * W * G) {
    re += p[0];
    im += p[G];
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
                                                   const int* nlive, int G, int W, double alpha, int nz) {
  k_fb_reduce_body(blockIdx3(), gridDim3(), part, fb, live, nlive, G, W, alpha, nz);
}

// Bound by FP64 MFMA issue.  K is long (Ktot = N (na + nb), 36,000 at N = 300, 60+60) and
// the output small (2W x G), so without a split of K a few tens of workgroups walk it
// serially: at N = 300, G = 1200, 256 walkers 40 workgroups took 12.5 ms (3.5 TFLOP/s); with
// K in 13 chunks it takes 0.80 ms (55 TFLOP/s) plus 18 us for the sum of the chunks.
// 64 x 64 tiles leave room for four workgroups on a CU, whose waves cover each other's
// barriers: 128 x 64 and 128 x 128 tiles took 0.82 and 1.02 ms there (0.080, 0.081, 0.095 ms
// at N = 100, G = 400, 512 walkers).  A grid of at most 64 such tiles gains from 32 x 64
// ones: 11 against 15 us for 16 determinants at N = 100, G = 400 (7 tiles), 15.0 against
// 17.4 us at N = 51, G = 205, 256 walkers (32 tiles); at 112 tiles (N = 100, 512 walkers)
// the 64 x 64 tile is ahead, 80 against 95 us.
// nz minimises the rounds of resident workgroups times the chunk's length (plus 64 for the
// prologue and epilogue of a chunk), within the borrowed workspace and chunks of 128.
FbPlan fb_plan(int W, int G, int64_t Ktot, int64_t ws_doubles) {
  FbPlan p;
  p.small = (int64_t)cdivu(G, 64) * cdivu(2 * (int64_t)W, 64) <= 64;
  const int64_t slots = p.small ? 1280 : 1024;   // resident workgroups: LDS allows 5 and 4 on a CU
  const int64_t tiles = (int64_t)cdivu(G, 64) * cdivu(2 * (int64_t)W, p.small ? 32 : 64);
  const int64_t most = std::max<int64_t>(1, std::min<int64_t>(Ktot / 128, ws_doubles / (2 * (int64_t)W * G)));
  int64_t best = INT64_MAX;
  p.nz = 1;
  p.kchunk = 0;
  for (int64_t nz = 1; nz <= most && nz <= 64; ++nz) {
    const int64_t kc = cdivu(cdivu(Ktot, nz), G64_BK) * G64_BK, z = cdivu(Ktot, kc);
    const int64_t cost = (int64_t)cdivu(tiles * z, slots) * (kc + 64);
    if (cost < best) {
      best = cost;
      p.nz = (int)z;
      p.kchunk = (int)kc;
    }
  }
  return p;
}

void launch_force_bias(const DevState& s, hipStream_t st) {
  launch_live_list(s, st);
  const FbPlan p = fb_plan(s.W, s.G, s.Ktot, s.fbw ? s.fbw_doubles : 0);
  const double alpha = (double)s.slot[0].mult;
  const int gx = (int)cdivu(s.G, 64), gy = (int)cdivu(2 * (int64_t)s.W, p.small ? 32 : 64);
  if (p.small)
    afq::glaunch<F_k_fb64<32, 64, 1, 4>>((k_fb64<32, 64, 1, 4>), dim3(gx * gy * p.nz), dim3(256), 0, st, s.R, s.theta, s.fb,
                                         s.fbw, s.live, s.nlive, s.G, s.W, s.Ktot, p.kchunk, alpha, gx, gy, p.nz);
  else
    afq::glaunch<F_k_fb64<64, 64, 2, 2>>((k_fb64<64, 64, 2, 2>), dim3(gx * gy * p.nz), dim3(256), 0, st, s.R, s.theta, s.fb,
                                         s.fbw, s.live, s.nlive, s.G, s.W, s.Ktot, p.kchunk, alpha, gx, gy, p.nz);
  if (p.nz > 1)
    afq::glaunch<F_k_fb_reduce>(k_fb_reduce, dim3(cdivu((int64_t)s.W * s.G, 256)), dim3(256), 0, st, s.fbw, s.fb, s.live,
                                s.nlive, s.G, s.W, alpha, p.nz);
}

}  // namespace afq
