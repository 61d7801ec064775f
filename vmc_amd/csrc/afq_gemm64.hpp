// FP64 MFMA block product with 16-byte operand loads, for the contractions whose
// operands lie in memory in one of two ways:
//   StageC  complex rows, K contiguous: element k of row pair (2w, 2w + 1) is one
//           (re, im) double2, so one 16-byte load feeds a real row and its imaginary twin
//   StageK  real rows, K contiguous: one 16-byte load holds two K of a row
// One stage is BK = 16 deep, double-buffered in LDS: stage s + 1 goes global ->
// registers before stage s is multiplied and registers -> LDS after it, one barrier a
// stage.  The K order inside a stage is 8 s + 2 (lane / 16) + {0, 1}, so that a lane of
// an operand reads the operands of two MFMAs with one ds_read_b128; rows of 18 doubles put
// the 16 lanes of such a read on 64 different banks.
#pragma once
#include "afq_device.hpp"

namespace afq {

// 16-byte load of two doubles that are only 8-byte aligned (odd offsets)
typedef double __attribute__((ext_vector_type(2), aligned(8))) f64x2u;
typedef double __attribute__((ext_vector_type(2))) f64x2;
__device__ __forceinline__ f64x2 load2(const double* p) {
  const f64x2u v = *reinterpret_cast<const f64x2u*>(p);
  return f64x2{v.x, v.y};
}

constexpr int G64_BK = 16;
constexpr int G64_LDK = G64_BK + 2;

// ROWS real rows = ROWS / 2 complex ones.  ptr(w): the complex row's element 0, or null
// (a row of zeros).  K: number of complex elements a row holds.
template <int ROWS, int NT>
struct StageC {
  static constexpr int SIZE = ROWS * G64_LDK;
  static constexpr int UNITS = ROWS / 2 * 8, U = (UNITS + NT - 1) / NT;   // (complex row, k pair)
  const double* p[U];
  f64x2 a[U], b[U];
  template <class P>
  __device__ __forceinline__ void init(const P& ptr) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = threadIdx.x + u * NT;
      p[u] = e < UNITS ? ptr(e >> 3) : nullptr;
      if (p[u]) p[u] += 4 * (e & 7);
    }
  }
  __device__ __forceinline__ void fetch(int k0, int kend) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 2 * ((threadIdx.x + u * NT) & 7);
      a[u] = f64x2{0.0, 0.0};
      b[u] = f64x2{0.0, 0.0};
      if (p[u] && k < kend) a[u] = load2(p[u] + 2 * (int64_t)k0);
      if (p[u] && k + 1 < kend) b[u] = load2(p[u] + 2 * (int64_t)k0 + 2);
    }
  }
  __device__ __forceinline__ void put(double* s) const {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = threadIdx.x + u * NT, kp = e & 7, w = e >> 3;
      if (UNITS % NT == 0 || e < UNITS) {
        *reinterpret_cast<f64x2*>(s + 2 * w * G64_LDK + 2 * kp) = f64x2{a[u].x, b[u].x};
        *reinterpret_cast<f64x2*>(s + (2 * w + 1) * G64_LDK + 2 * kp) = f64x2{a[u].y, b[u].y};
      }
    }
  }
  __device__ __forceinline__ static f64x2 frag(const double* s, int row, int kq) {
    return *reinterpret_cast<const f64x2*>(s + row * G64_LDK + kq);
  }
};

// ROWS real rows.  ptr(r): the row's element 0, or null (a row of zeros).
template <int ROWS, int NT>
struct StageK {
  static constexpr int SIZE = ROWS * G64_LDK;
  static constexpr int UNITS = ROWS * 8, U = (UNITS + NT - 1) / NT;   // (row, k pair)
  const double* p[U];
  f64x2 a[U];
  template <class P>
  __device__ __forceinline__ void init(const P& ptr) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = threadIdx.x + u * NT;
      p[u] = e < UNITS ? ptr(e >> 3) : nullptr;
      if (p[u]) p[u] += 2 * (e & 7);
    }
  }
  __device__ __forceinline__ void fetch(int k0, int kend) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 2 * ((threadIdx.x + u * NT) & 7);
      a[u] = f64x2{0.0, 0.0};
      if (p[u] && k + 1 < kend) a[u] = load2(p[u] + k0);
      else if (p[u] && k < kend) a[u].x = p[u][k0];
    }
  }
  __device__ __forceinline__ void put(double* s) const {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = threadIdx.x + u * NT, kp = e & 7, r = e >> 3;
      if (UNITS % NT == 0 || e < UNITS) *reinterpret_cast<f64x2*>(s + r * G64_LDK + 2 * kp) = a[u];
    }
  }
  __device__ __forceinline__ static f64x2 frag(const double* s, int row, int kq) {
    return *reinterpret_cast<const f64x2*>(s + row * G64_LDK + kq);
  }
};

// C += A B for a BM x BN tile over K in [k0, kend), k0 a multiple of 16; waves WM x WN.  At the
// end of every ku of K (a multiple of 16) and of the last, shorter one, unit(acc) is called, and
// acc starts from zero again.
template <class SA, class SB, int BM, int BN, int WAVES_M, int WAVES_N>
struct Gemm64 {
  static constexpr int NT = 64 * WAVES_M * WAVES_N;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, TM = WM / 16, TN = WN / 16;
  static constexpr int STAGE = SA::SIZE + SB::SIZE, LDS_DOUBLES = 2 * STAGE;
  static_assert(WM % 16 == 0 && WN % 16 == 0, "wave tile must be a multiple of 16");
  f64x4 acc[TM][TN];
  int lane, wm, wn;
  __device__ __forceinline__ Gemm64() {
    lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    wm = wave / WAVES_N;
    wn = wave % WAVES_N;
    clear();
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
  }
  template <class U>
  __device__ __forceinline__ void run(SA& sa, SB& sb, int k0, int kend, double* lds, int ku, const U& unit) {
    if (k0 >= kend) return;
    int uend = k0 + ku;
    sa.fetch(k0, kend);
    sb.fetch(k0, kend);
    sa.put(lds);
    sb.put(lds + SA::SIZE);
    __syncthreads();
    int buf = 0;
    for (int k = k0; k < kend; k += G64_BK) {
      const bool more = k + G64_BK < kend;
      if (more) {
        sa.fetch(k + G64_BK, kend);
        sb.fetch(k + G64_BK, kend);
      }
      const double* As = lds + buf * STAGE;
      const double* Bs = As + SA::SIZE;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kq = 8 * h + 2 * (lane >> 4);
        f64x2 a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = SA::frag(As, wm * WM + i * 16 + (lane & 15), kq);
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = SB::frag(Bs, wn * WN + j * 16 + (lane & 15), kq);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b[j].x, acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].y, b[j].y, acc[i][j], 0, 0, 0);
      }
      buf ^= 1;
      if (more) {
        sa.put(lds + buf * STAGE);
        sb.put(lds + buf * STAGE + SA::SIZE);
      }
      if (!more || k + G64_BK == uend) {
        unit(acc);
        clear();
        uend += ku;
      }
      __syncthreads();
    }
  }
  // tile-relative coordinates of accumulator element acc[i][j][r]
  __device__ __forceinline__ int row(int i, int r) const { return wm * WM + i * 16 + (lane >> 4) + 4 * r; }
  __device__ __forceinline__ int col(int j) const { return wn * WN + j * 16 + (lane & 15); }
  template <class EP>
  __device__ __forceinline__ void store(const f64x4 (&v)[TM][TN], const EP& ep) const {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) ep(row(i, r), col(j), v[i][j][r]);
  }
};

}  // namespace afq
