// Two of the three kernels of the Green's function (see launch_green_pre, launch_theta_post):
// the overlap matrices S = Phi^T psi and theta = psi S^-1.  Both read their memory operands
// straight into FP64 MFMA registers a few K steps ahead, so neither K loop has a barrier.
#include <algorithm>

#include "afq_device.hpp"
#include "afq_internal.hpp"

namespace afq {

static inline unsigned cdivu(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

// S = Phi_s^T psi of every walker of a slot as one product over the W n complex columns
// (walker, electron): a wave takes 16 columns (one 16-byte load of a lane is re and im, the B
// operands of two MFMA tiles) against all n <= 64 rows (trial orbitals).  grid.y: slot.
// Both spins of 4096 walkers at N = 300, 60+60: 0.70 ms (50 TFLOP/s; 0.83 as 64 x 128 tiles
// through LDS with an element loader); of 1024 walkers at N = 100, 20+20: 23 us (53).
__device__ __forceinline__ void k_overlap_body(const uint3 bid_, const uint3 gdim_, GreenArgs a) {
  constexpr int NS = 4;
  const int si = bid_.y;
  const Slot sl = si == 0 ? a.s0 : a.s1;
  const int n = sl.n, N = a.N, lane = threadIdx.x & 63, cl = lane & 15, kh = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t ncol = (int64_t)a.W * n, q0 = (int64_t)bid_.x * 64 + 16 * wave;
  if (q0 >= ncol) return;
  const int64_t q = min(q0 + cl, ncol - 1);   // columns past the last read a valid one
  const int w = (int)(q / n), j = (int)(q - (int64_t)w * n);
  const double* pb = a.psi + (int64_t)w * 2 * a.ms + 2 * (sl.det == 0 ? a.det_off0 : a.det_off1) + 2 * j;
  const double* phi = sl.phi == 0 ? a.phi0 : a.phi1;
  int ro[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) ro[i] = min(16 * i + cl, n - 1);
  const int rt = (n + 15) >> 4, nk = (N + 3) >> 2;
  double A[NS][4];
  double2 B[NS];
  auto load = [&](int s, int set) {
    const int k = min(4 * s + kh, N - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) A[set][i] = phi[k * n + ro[i]];
    B[set] = *reinterpret_cast<const double2*>(pb + (int64_t)k * 2 * n);
  };
  f64x4 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i][0] = acc[i][1] = f64x4{0.0, 0.0, 0.0, 0.0};
  auto step = [&](int set) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i >= rt) continue;   // uniform
      acc[i][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set][i], B[set].x, acc[i][0], 0, 0, 0);
      acc[i][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set][i], B[set].y, acc[i][1], 0, 0, 0);
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
  // the last one to NS steps (NS - 1 of them requested); k past N add nothing
  if (s + NS - 1 < nk) load(s + NS - 1, NS - 1);
#pragma unroll
  for (int i = 0; i < NS; ++i)
    if (s + i < nk) {
      if (4 * (s + i) + kh >= N) B[i] = double2{0.0, 0.0};
      step(i);
    }
  if (q0 + cl >= ncol || (!a.all && a.weights[w] <= 1e-8)) return;
  double* S = a.Sg + ((int64_t)w * a.nslots + si) * SG_MAT + 2 * j;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * i + kh + 4 * r;
      if (row < n) *reinterpret_cast<double2*>(S + row * SG_LD) = double2{acc[i][0][r], acc[i][1][r]};
    }
}
struct F_k_overlap {
  static constexpr int NT = 256, OCC = 3;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_overlap_body(b, g, a...);
  }
};
__global__ __launch_bounds__(256, 3) void k_overlap(GreenArgs a) { k_overlap_body(blockIdx3(), gridDim3(), a); }

void launch_overlap(const GreenArgs& a, hipStream_t st) {
  const int nmax = std::max(a.s0.n, a.nslots > 1 ? a.s1.n : 0);
  afq::glaunch<F_k_overlap>(k_overlap, dim3(cdivu((int64_t)a.W * nmax, 64), a.nslots), dim3(256), 0, st, a);
}

// theta = psi S^-1 of one (walker, slot), n <= 8 CT, and the one-body partial
// e1 = sum theta o (h1 Phi).  S^-1 lies in LDS as [k][re, im interleaved], the B operand: the
// complex product is psi_re against column c and psi_im against its neighbour c ^ 1, negated
// in the real columns.  Four waves take the row tiles (16 orbitals) in turn; a lane's 16-byte
// load of psi is the A operand of both.  Row 4 (c % 4) + c / 4 of the tile sits in lane c, so
// that a lane ends with four consecutive orbitals of its column, which the split copy of
// theta (tbh, tbl: k contiguous) stores as 8 bytes.
// Bound by reading psi and writing theta as much as by MFMA issue.  CT follows n, where a form
// with S^-1 in registers padded every n to 64: 1024 walkers at N = 100, 20+20 195 -> 41 us;
// 256 at N = 300, 60+60 137 -> 116 us; 4096 there with the split copy 2.50 -> 2.15 ms.
template <int CT>
__device__ __forceinline__ void k_theta_body(const uint3 bid_, const uint3 gdim_, GreenArgs a) {
  constexpr int NS = 4, LD = 16 * CT, KR = 8 * CT;
  __shared__ __attribute__((aligned(16))) double Ss[KR * LD];
  __shared__ double red[16];
  const int w = bid_.x, si = bid_.y;
  if (a.post ? (!a.fresh[w] || a.weights[w] == 0.0) : (!a.all && a.weights[w] <= 1e-8)) return;
  const Slot sl = si == 0 ? a.s0 : a.s1;
  const int n = sl.n, N = a.N, n2 = 2 * n, nk = (n + 3) >> 2;
  const int tid = threadIdx.x, lane = tid & 63, cl = lane & 15, kh = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const double* psi = a.psi + (int64_t)w * 2 * a.ms + 2 * (sl.det == 0 ? a.det_off0 : a.det_off1);
  const double* hphi = sl.phi == 0 ? a.hphi0 : a.hphi1;
  const double* Si = a.Sg + ((int64_t)w * a.nslots + si) * SG_MAT;
  double* th = a.theta + (int64_t)w * 2 * a.Ktot + 2 * sl.koff;
  const int RT = (N + 15) >> 4, nt = (RT - wave + 3) >> 2;   // row tiles; this wave's (tiles wave, wave + 4, ..)
  const int rperm = 4 * (cl & 3) + (cl >> 2);
  double2 A[NS];
  // step s of this wave's tile sequence: K step s % nk of its tile s / nk
  int lt = 0, lk = 0;   // the step requested next
  auto load = [&](int set) {
    const int row = min(16 * (wave + 4 * lt) + rperm, N - 1), k = min(4 * lk + kh, n - 1);
    A[set] = *reinterpret_cast<const double2*>(psi + 2 * ((int64_t)row * n + k));
    if (++lk == nk) { lk = 0; ++lt; }
  };
#pragma unroll
  for (int i = 0; i + 1 < NS; ++i) load(i);
  for (int e = tid; e < 4 * nk * LD; e += 256) {
    const int k = e / LD, c = e - k * LD;
    const double v = k < n && c < n2 ? Si[k * SG_LD + c] : 0.0;
    Ss[k * LD + (CT % 2 == 0 ? c ^ ((k & 1) << 4) : c)] = v;   // odd k swap column tiles 2 i and 2 i + 1 (banks)
  }
  __syncthreads();
  const int sw = CT % 2 == 0 ? 16 * (kh & 1) : 0;
  auto at = [&](int j, int c) { return 16 * j + (j & 1 ? c - sw : c + sw); };
  const unsigned flip = (cl & 1) ? 0u : 0x80000000u;
  f64x4 acc[CT];
  double e1re = 0.0, e1im = 0.0;
  auto step = [&](int ks, int set) {
    const double* S = Ss + (4 * ks + kh) * LD;
    double b1[CT], b2[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      b1[j] = S[at(j, cl)];
      const double v = S[at(j, cl ^ 1)];
      b2[j] = __hiloint2double(__double2hiint(v) ^ flip, __double2loint(v));
    }
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set].x, b1[j], acc[j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[set].y, b2[j], acc[j], 0, 0, 0);
  };
  auto clear = [&]() {
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[j] = f64x4{0.0, 0.0, 0.0, 0.0};
  };
  // h1 Phi at a tile's output positions, requested before the tile's last K step: a load
  // behind the stores of theta would wait for them (one counter for both)
  double hv[CT][4];
  auto hload = [&](int tile) {
    const int row0 = 16 * tile + 4 * kh;
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) hv[j][r] = hphi[min(row0 + r, N - 1) * n + min((16 * j + cl) >> 1, n - 1)];
  };
  auto store = [&](int tile) {
    const int row0 = 16 * tile + 4 * kh;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int c = 16 * j + cl;
      if (c >= n2) continue;
      u16 hb[4], lb[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = row0 + r;
        const double v = row < N ? acc[j][r] : 0.0;
        if (row < N) {
          th[(int64_t)row * n2 + c] = v;
          if (c & 1) e1im += v * hv[j][r];
          else e1re += v * hv[j][r];
        }
        if (a.tbh) split_bf16(v, hb[r], lb[r]);
      }
      if (a.tbh && row0 < a.Np) {   // pad rows N .. Np - 1 are zero; Np is a multiple of 8
        const int64_t ta = (((int64_t)w * 2 + (c & 1)) * (a.ctot / 2) + (si == 0 ? 0 : a.s0.n) + (c >> 1)) * a.Np + row0;
        *reinterpret_cast<uint2*>(a.tbh + ta) = uint2{hb[0] | (unsigned)hb[1] << 16, hb[2] | (unsigned)hb[3] << 16};
        *reinterpret_cast<uint2*>(a.tbl + ta) = uint2{lb[0] | (unsigned)lb[1] << 16, lb[2] | (unsigned)lb[3] << 16};
      }
    }
  };
  clear();
  int tile = 0, ks = 0;
  for (int s = 0; s < nt * nk; s += NS) {
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      if (s + i >= nt * nk) break;
      load((i + NS - 1) % NS);
      if (ks == nk - 1) hload(wave + 4 * tile);
      step(ks, i);
      if (++ks == nk) {
        store(wave + 4 * tile);
        clear();
        ks = 0;
        ++tile;
      }
    }
  }
  e1re = block_sum(e1re, red);
  e1im = block_sum(e1im, red);
  if (tid == 0) {
    a.e1[2 * ((int64_t)w * a.nslots + si)] = e1re;
    a.e1[2 * ((int64_t)w * a.nslots + si) + 1] = e1im;
  }
}
template <int CT>
struct F_k_theta {
  static constexpr int NT = 256, OCC = CT > 4 ? 2 : 3;
  static constexpr bool HAS_OCC = true;
  template <class... A>
  __device__ __forceinline__ void operator()(const uint3 b, const uint3 g, A... a) const {
    k_theta_body<CT>(b, g, a...);
  }
};
template <int CT>
__global__ __launch_bounds__(256, CT > 4 ? 2 : 3) void k_theta(GreenArgs a) {
  k_theta_body<CT>(blockIdx3(), gridDim3(), a);
}

void launch_theta(const GreenArgs& a, hipStream_t st) {
  const dim3 grid(a.W, a.nslots);
  const int nmax = std::max(a.s0.n, a.nslots > 1 ? a.s1.n : 0);
#define AFQ_THETA(CT_)                                                            \
  case CT_:                                                                       \
    afq::glaunch<F_k_theta<CT_>>((k_theta<CT_>), grid, dim3(256), 0, st, a); \
    break
  switch ((nmax + 7) / 8) {
    AFQ_THETA(1);
    AFQ_THETA(2);
    AFQ_THETA(3);
    AFQ_THETA(4);
    AFQ_THETA(5);
    AFQ_THETA(6);
    AFQ_THETA(7);
    AFQ_THETA(8);
  }
#undef AFQ_THETA
}

}  // namespace afq
