// FP64 exchange: Xp[s][w][tile] = sum over a tile of Cholesky vectors g of
// sum_ij f_ij f_ji, f = R_{s,g} theta_s (DQMC/UHF.cpp:94-100), without writing f to memory.
#include <algorithm>

#include "afq_device.hpp"
#include "afq_internal.hpp"

namespace afq {

static inline unsigned cdivu(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

// One workgroup (WAVES of them, 4 or 3) takes gt = 64 / n walkers of a slot and a chunk of the
// Cholesky vectors, gt at a time: the tile's rows are (vector, i), at most 16 WAVES, its columns
// (walker, j), at most 16 WAVES complex ones, 16 for each wave.  Both operands go from global
// memory straight into MFMA registers, NS - 1 K steps of 4 ahead: one 16-byte load of a lane
// holds re and im of a theta column (the B operands of two MFMA tiles), and for even n two
// rows of R_g (the A operands of two tiles: rows 2 l of 32 in one, 2 l + 1 in the other; for
// odd n, where a pair of rows may belong to two vectors, two 8-byte loads).  The waves of a
// workgroup share the R lines in the vector L1, and without staging the K loop has no
// barrier.  f then goes to LDS and the sum runs over i <= j (off-diagonal pairs count
// twice), so that every element of f is read once.  A group of tpb threads keeps the same
// (vector, walker) place of the tile and accumulates in registers.
//
// The vectors fall into units of uv (a multiple of gt), a chunk being whole units, and at a unit's
// end one wave adds up its sum into its own partial (the walker's further partials are zero).  Units
// depend on n and on the vectors in the energy alone, never on how many walkers are taken together,
// which decides only how many units a chunk has: so a walker's exchange is the same to the last bit in
// any company.  Against one sum for a whole chunk: N = 300, 60+60, 256 walkers 48.2 against 48.0 ms,
// N = 100, 20+20, 1024 walkers 2.82 both, N = 160, 40+40, 128 walkers 4.66 against 4.48 (units divide
// the chunks less evenly), N = 51, 13+11, 256 walkers 0.165 against 0.151; with the sum as a tree over
// the workgroup's threads behind barriers 2.91 at N = 100.
//
// Bound by FP64 MFMA issue.  N = 300, 60+60, G = 1200, 256 walkers: 53.4 ms on the 128 x 128
// LDS-staged kernel before, 48.2 now (55 TFLOP/s useful, 64 with the padding of 60 to 64;
// 46.0 of it the K loops, timed without the pair sums).  N = 100, 20+20, G = 400, 1024
// walkers: 3.8 -> 2.82 ms (47 TFLOP/s; K loops 2.54).  A form with LDS stages of both
// operands took 56 and 3.3 ms (two 8-byte LDS reads per MFMA), one with 8-byte global loads
// per tile 49.2 and 3.06.  NS = 6 against 4: equal at N = 100 and 300, 3% faster on systems of
// N = 20 to 120.
template <int WAVES>
struct X64Shape {
  static constexpr int NT = 64 * WAVES, ROWS = 16 * WAVES, OCC = WAVES == 4 ? 2 : 3;
  static constexpr int LDF = 2 * ROWS + 2;   // 16-byte rows; transposed 16-byte reads of 16 lanes on 64 banks
};
typedef double __attribute__((ext_vector_type(2), aligned(8))) x64_pair;   // two rows of R, 8-byte aligned
// x of the lane that DPP control CTRL names
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
  const int hi = __double2hiint(x), lo = __double2loint(x);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xF, 0xF, false),
                          __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xF, 0xF, false));
}
template <bool EVEN, int WAVES>
__device__ __forceinline__ void k_exchange64_body(const uint3 bid_, const uint3 gdim_, const double* R, const double* theta,
                                                  const int* sel, const int* nsel_dev, double* Xp, int N, int GE, int nw,
                                                  int W, int64_t Ktot, Slot s0, Slot s1, int ngt_cap, int nt, int uv, int nu, int upc,
                                                  int gridx, int gridy, int gridz) {
  constexpr int NS = 6, NT = X64Shape<WAVES>::NT, LDF = X64Shape<WAVES>::LDF;
  __shared__ __attribute__((aligned(16))) double lds[X64Shape<WAVES>::ROWS * LDF];
  __shared__ double2 red[NT];
  __shared__ int walker[16];
  const TileId tl = tile_id_at(bid_.x, gridx, gridy, gridz, 8);
  const Slot sl = tl.z == 0 ? s0 : s1;
  const int n = sl.n, gt = 64 / n, w0 = tl.y * gt, nrow = gt * n;
  if (nsel_dev) nw = *nsel_dev;
  if (w0 >= nw) return;
  const int ga = tl.x * upc * uv, gb = min(GE, ga + upc * uv);   // this chunk's vectors, units tl.x upc .. + upc - 1
  const int tid = threadIdx.x, lane = tid & 63, cl = lane & 15, kh = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < gt) walker[tid] = w0 + tid >= nw ? -1 : sel ? sel[w0 + tid] : w0 + tid;
  const bool busy = 16 * wave < nrow;   // this wave's columns hold data
  // rows 32 .. nrow (gt n > 32 always): as two tiles, or as one where at most 16 (row 32 + cl)
  const int rest = nrow - 32;
  const bool two1 = WAVES == 4 && rest > 16;
  // A: rows past the data read a valid one
  auto split = [&](int r, int& g, int& e) {
    r = min(r, nrow - 1);
    g = r / n;
    e = r - g * n;
  };
  int ag[2][2], ae[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    split(2 * cl + t, ag[0][t], ae[0][t]);
    split(two1 ? 32 + min(2 * cl, EVEN ? rest - 2 : rest) + t : 32 + cl, ag[1][t], ae[1][t]);   // an even n's pair stays one
  }
  // B: complex column 16 wave + cl = (walker, j); columns past the data read a valid one
  const double* pb;
  {
    const int c = min(16 * wave + cl, nrow - 1), wl = c / n, j = c - wl * n;
    const int wi = w0 + wl < nw ? w0 + wl : w0;
    const int w = sel ? sel[wi] : wi;
    pb = theta + (int64_t)w * 2 * Ktot + 2 * sl.koff + 2 * j;
  }
  const double* Rs = R + sl.koff;
  const int nk = (N + 3) >> 2;
  const double* pa[2][2];
  double2 A[NS][2], B[NS];
  auto rows = [&](int g0) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < 2; ++t) pa[h][t] = Rs + (int64_t)min(g0 + ag[h][t], GE - 1) * Ktot + ae[h][t];
  };
  auto load = [&](int s, int set) {
    const int k = min(4 * s + kh, N - 1);
    auto two = [&](int h) {
      if (EVEN) {
        const x64_pair v = *reinterpret_cast<const x64_pair*>(pa[h][0] + k * n);
        A[set][h] = double2{v.x, v.y};
      } else {
        A[set][h].x = pa[h][0][k * n];
        A[set][h].y = pa[h][1][k * n];
      }
    };
    two(0);
    if (two1) two(1);
    else A[set][1].x = pa[1][0][k * n];
    B[set] = *reinterpret_cast<const double2*>(pb + k * 2 * n);
  };
  f64x4 acc[2][2][2];   // [32 rows][even, odd][re, im]
  auto step = [&](int set) {
    if (!busy) return;
    acc[0][0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set][0].x, B[set].x, acc[0][0][0], 0, 0, 0);
    acc[0][0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set][0].x, B[set].y, acc[0][0][1], 0, 0, 0);
    acc[0][1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set][0].y, B[set].x, acc[0][1][0], 0, 0, 0);
    acc[0][1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set][0].y, B[set].y, acc[0][1][1], 0, 0, 0);
    acc[1][0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set][1].x, B[set].x, acc[1][0][0], 0, 0, 0);
    acc[1][0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set][1].x, B[set].y, acc[1][0][1], 0, 0, 0);
    if (two1) {
      acc[1][1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set][1].y, B[set].x, acc[1][1][0], 0, 0, 0);
      acc[1][1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set][1].y, B[set].y, acc[1][1][1], 0, 0, 0);
    }
  };
  // pair sums: threads [b tpb, (b + 1) tpb) take block b = (vector b / gt, walker b % gt) of a tile
  const int tpb = NT / (gt * gt), rtpb = 65536 / tpb + 1;
  const int blk = tid / tpb, lt = tid - blk * tpb, pg = blk / gt, pw = blk - pg * gt;
  // units (p, t): rows p and n - 1 - p share the n + 1 pairs i <= j
  const int np = (n + 1) >> 1, sp = tpb / (n + 1), stt = tpb - sp * (n + 1);
  int place = pw << 24 | pg << 16 | (lt / (n + 1)) << 8 | lt % (n + 1);   // one register through the K loops
  // the lane's number asked for again, so that no register holds it or an address through the K loops
  auto lane_again = [] {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
  };
  double accr = 0.0, acci = 0.0;
  rows(ga);
#pragma unroll
  for (int i = 0; i + 1 < NS; ++i) load(i, i);
  int unit = tl.x * upc, ub = min(gb, ga + uv);   // the unit at hand and its end
  for (int g0 = ga; g0 < gb;) {
    const int gn = min(g0 + gt, ub);   // the next tile's first vector
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[h][t][0] = acc[h][t][1] = f64x4{0.0, 0.0, 0.0, 0.0};
    int s = 0;
    for (; s + NS < nk; s += NS) {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        load(s + i + NS - 1, (i + NS - 1) % NS);
        step(i);
      }
    }
    // the last one to NS steps (NS - 1 of them requested); k past N add nothing
    if (s + NS - 1 < nk) load(s + NS - 1, NS - 1);
#pragma unroll
    for (int i = 0; i < NS; ++i)
      if (s + i < nk) {
        if (4 * (s + i) + kh >= N) B[i] = double2{0.0, 0.0};
        step(i);
      }
    // the next tile's first steps are in flight during the pair sums
    rows(gn);
#pragma unroll
    for (int i = 0; i + 1 < NS; ++i) load(i, i);
    if (busy) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          if (h == 1 && t == 1 && !two1) continue;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int d = kh + 4 * r, row = h == 0 ? 2 * d + t : 32 + (two1 ? 2 * d + t : d);
            *reinterpret_cast<double2*>(lds + row * LDF + 2 * (16 * wave + cl)) =
                double2{acc[h][t][0][r], acc[h][t][1][r]};
          }
        }
    }
    __syncthreads();
    asm volatile("" : "+v"(place));
    if ((place >> 16 & 255) < min(gt, gn - g0)) {
      const double* F = lds + (place >> 16 & 255) * n * LDF + (place >> 24) * 2 * n;
      int p = place >> 8 & 255, t = place & 255;
      while (p < np) {
        const bool first = t < n - p;
        const int i = first ? p : n - 1 - p, j = first ? p + t : t - 1;   // second row: j = i + t - (n - p)
        if (first || 2 * p != n - 1) {
          const double2 x = *reinterpret_cast<const double2*>(F + i * LDF + 2 * j);
          const double2 y = *reinterpret_cast<const double2*>(F + j * LDF + 2 * i);
          const double m = i == j ? 1.0 : 2.0;
          accr += m * (x.x * y.x - x.y * y.y);
          acci += m * (x.x * y.y + x.y * y.x);
        }
        p += sp;
        t += stt;
        if (t > n) { t -= n + 1; ++p; }
      }
    }
    if (gn == ub) {
      red[64 * wave + lane_again()] = double2{accr, acci};
      accr = acci = 0.0;
    }
    __syncthreads();
    g0 = gn;
    if (g0 < ub) continue;
    ub = min(gb, ub + uv);
    // the unit's sum by one wave while the others go on: 2^sh lanes a walker take its gt tpb threads'
    // sums in turn (at most 7 each), then a tree over the lanes.  (red is written again only behind the
    // next tile's barriers.)
    if (wave == 0) {
      const int lq = lane_again();
      int sh = 6;
      while (gt << sh > 64) --sh;
      const int q = lq >> sh, sub = lq & ((1 << sh) - 1), ne = q < gt ? gt * tpb : 0;
      double xr = 0.0, xi = 0.0;
#pragma unroll
      for (int i = 0; i < 7; ++i) {
        const int e = sub + (i << sh), g = e * rtpb >> 16;   // e / tpb for e < 256
        if (e < ne) {
          const double2 x = red[(g * gt + q) * tpb + e - g * tpb];
          xr += x.x;
          xi += x.y;
        }
      }
      if (sh >= 5) {
        for (int off = 1 << (sh - 1); off >= 16; off >>= 1) {
          xr += __shfl_xor(xr, off, 64);
          xi += __shfl_xor(xi, off, 64);
        }
      }
      if (sh >= 4) xr += dpp_f64<0x140>(xr), xi += dpp_f64<0x140>(xi);   // row_mirror
      if (sh >= 3) xr += dpp_f64<0x141>(xr), xi += dpp_f64<0x141>(xi);   // row_half_mirror
      xr += dpp_f64<0x4E>(xr), xi += dpp_f64<0x4E>(xi);                  // quad_perm [2,3,0,1]
      xr += dpp_f64<0xB1>(xr), xi += dpp_f64<0xB1>(xi);                  // quad_perm [1,0,3,2]
      const int w = sub == 0 && q < gt ? walker[q] : -1;
      if (w >= 0) {
        double2* o = reinterpret_cast<double2*>(Xp) + ((int64_t)tl.z * W + w) * ngt_cap;
        o[unit] = double2{xr, xi};
        for (int t = unit + nu; t < nt; t += nu) o[t] = double2{0.0, 0.0};
      }
    }
    ++unit;
  }
}
template <bool EVEN, int WAVES>
struct F_k_exchange64 {
  static constexpr int NT = 64 * WAVES, OCC = WAVES == 4 ? 2 : 3;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_exchange64_body<EVEN, WAVES>(b, g, a...);
  }
};
template <bool EVEN, int WAVES>
__global__ __launch_bounds__(64 * WAVES, WAVES == 4 ? 2 : 3) void k_exchange64(const double* R, const double* theta, const int* sel,
                                                          const int* nsel_dev, double* Xp, int N, int GE, int nw, int W,
                                                          int64_t Ktot, Slot s0, Slot s1, int ngt_cap, int nt, int uv, int nu, int upc,
                                                          int gridx, int gridy, int gridz) {
  k_exchange64_body<EVEN, WAVES>(blockIdx3(), gridDim3(), R, theta, sel, nsel_dev, Xp, N, GE, nw, W, Ktot, s0, s1, ngt_cap, nt, uv, nu,
                          upc, gridx, gridy, gridz);
}

// slots a and b (b of a's size; nz = 1: a alone), partials at xp
void launch_exchange64(const DevState& s, const int* sel, int nsel, const int* nsel_dev, double* xp, Slot a, Slot b, int nz,
                       hipStream_t st) {
  // units of the vectors: whole tiles, no more units than there are partials, and 64 at most (a unit
  // costs about 900 cycles of one wave, 3 % with units of two tiles at N = 100)
  const int gslot = exchange_tile_g(a.n), gt = 64 / a.n, nt = (int)cdivu(s.GE, gslot), gy = (int)cdivu(nsel, gt);
  const int u1 = (int)cdivu(gslot, gt) * gt, uv = u1 * (int)cdivu(cdivu(s.GE, u1), 64), nu = (int)cdivu(s.GE, uv);
  // gt n rows and columns fill 44 to 48 at n = 22 to 24 and 33 to 48 with one walker a tile: the
  // fourth wave would have no columns there, and a tile of 48 leaves registers and LDS for four
  // workgroups on a CU instead of two.  N = 100, G = 400, 1024 walkers, n = 23: 4.75 ms with four
  // waves, 3.73 with three; n = 24 4.68 and 3.65; N = 300, n = 40 and 45, 128 walkers 9.3 and 8.4.
  const bool three = gt * a.n <= 48;
  const int slots = three ? 1024 : 512;   // resident workgroups
  // chunks of units: at least 8 where there are as many, so that the resident workgroups of an XCD
  // (8 walker tiles x 8 chunks, tile_id_at) keep their theta in its L2 while R streams; among those
  // the fewest rounds of resident workgroups
  int upc = nu;
  int64_t best = INT64_MAX;
  for (int nc = std::min(8, nu); nc <= nu; ++nc) {
    const int per = (int)cdivu(nu, nc), z = (int)cdivu(nu, per);
    const int64_t cost = (int64_t)cdivu((int64_t)z * gy * nz, slots) * (2 * (int64_t)per * (uv / gt) + 1);
    if (cost < best) {
      best = cost;
      upc = per;
    }
  }
  const int nx = (int)cdivu(nu, upc);
#define AFQ_X64(EVEN_, WAVES_)                                                                                        \
  afq::glaunch<F_k_exchange64<EVEN_, WAVES_>>((k_exchange64<EVEN_, WAVES_>), dim3((unsigned)(nx * gy * nz)), dim3(64 * WAVES_), \
                                              0, st, s.R, s.theta, sel, nsel_dev, xp, s.N, s.GE, nsel, s.W, s.Ktot, a, b,        \
                                              s.ngt_cap, nt, uv, nu, upc, nx, gy, nz)
  if (a.n % 2 == 0) {
    if (three) AFQ_X64(true, 3);
    else AFQ_X64(true, 4);
  } else {
    if (three) AFQ_X64(false, 3);
    else AFQ_X64(false, 4);
  }
#undef AFQ_X64
}

}  // namespace afq
