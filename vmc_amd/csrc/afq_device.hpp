// Device building blocks for the CDNA4 (gfx950) phaseless-AFQMC kernels.
//
//  * MmaF64: a block-level FP64 MFMA tile engine.  One workgroup of
//    64*WAVES_M*WAVES_N threads computes a BM x BN tile of C = A * B where the
//    operands are produced element-wise by loader functors (so packed, strided,
//    gathered or complex-embedded operands all become plain real GEMMs), staged
//    through LDS in BK=16 slices with one slice of register prefetch, and
//    accumulated with v_mfma_f64_16x16x4_f64.
//  * small complex helpers and wavefront / block reductions (64-wide waves).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "afq_group.hpp"

namespace afq {

typedef double __attribute__((ext_vector_type(4))) f64x4;
typedef float __attribute__((ext_vector_type(4))) f32x4;

struct cplx {
  double re, im;
};
__device__ __forceinline__ cplx cmul(cplx a, cplx b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ __forceinline__ cplx cadd(cplx a, cplx b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ cplx csub(cplx a, cplx b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ cplx cscale(cplx a, double s) { return {a.re * s, a.im * s}; }
__device__ __forceinline__ cplx cdiv(cplx a, cplx b) {
  // Smith's algorithm
  if (fabs(b.re) >= fabs(b.im)) {
    const double r = b.im / b.re, d = b.re + b.im * r;
    return {(a.re + a.im * r) / d, (a.im - a.re * r) / d};
  }
  const double r = b.re / b.im, d = b.im + b.re * r;
  return {(a.re * r + a.im) / d, (a.im * r - a.re) / d};
}
__device__ __forceinline__ cplx clog(cplx a) { return {log(hypot(a.re, a.im)), atan2(a.im, a.re)}; }
__device__ __forceinline__ cplx cexp(cplx a) {
  const double m = exp(a.re);
  double s, c;
  sincos(a.im, &s, &c);
  return {m * c, m * s};
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// lane l's value in every lane (l uniform)
__device__ __forceinline__ double readlane_f64(double x, int l) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as easy as 1, 2,
// 3", SC'11): counter-based, so every (key, counter) pair gives its own 128 random bits.
__device__ __host__ inline void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
  for (int i = 0; i < 10; ++i) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
    const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
    const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
    c[0] = n0; c[1] = (uint32_t)p1; c[2] = n2; c[3] = (uint32_t)p0;
    k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
  }
}

// Sum over the whole block (blockDim.x multiple of 64, <= 1024).  All threads
// receive the result.  scratch: >= 16 doubles of LDS.
__device__ __forceinline__ double block_sum(double v, double* scratch) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  double t = 0.0;
  for (int i = 0; i < nw; ++i) t += scratch[i];
  __syncthreads();
  return t;
}

// ---------------------------------------------------------------------------
// Tile scheduling.  Kernels launch a 1-D grid of nx*ny*nz workgroups; the
// hardware deals consecutive workgroup ids round-robin over the 8 XCDs (each
// with its own L2).  tile_id() first makes each XCD's share a contiguous range
// of logical ids, then walks (x, y) in groups of `gy` rows along y (y fastest
// inside a group) so that the workgroups resident on one XCD at a time share
// both their A and their B operand tiles in that XCD's L2; z is slowest.
// ---------------------------------------------------------------------------
constexpr unsigned kXCDs = 8;
struct TileId {
  int x, y, z;
};
// b: the workgroup's index in the launch's 1-D grid (blockIdx.x for a plain launch)
__device__ __forceinline__ TileId tile_id_at(unsigned b, int nx, int ny, int nz, int gy) {
  const unsigned total = (unsigned)nx * ny * nz;
  const unsigned per = total / kXCDs;
  const unsigned pid = (b < per * kXCDs) ? (b % kXCDs) * per + b / kXCDs : b;
  const unsigned per_z = (unsigned)nx * ny;
  const int z = (int)(pid / per_z);
  const unsigned p = pid - (unsigned)z * per_z;
  const unsigned gsz = (unsigned)gy * nx;
  const unsigned grp = p / gsz;
  const int y0 = (int)(grp * gy);
  const int ysz = min(ny - y0, gy);
  const unsigned r = p - grp * gsz;
  TileId t;
  t.y = y0 + (int)(r % ysz);
  t.x = (int)(r / ysz);
  t.z = z;
  return t;
}
__device__ __forceinline__ TileId tile_id(int nx, int ny, int nz, int gy) {
  return tile_id_at(blockIdx.x, nx, ny, nz, gy);
}

// ---------------------------------------------------------------------------
// FP64 MFMA tile engine.
//
// v_mfma_f64_16x16x4_f64 operand layout (one 64-lane wave):
//   A (16x4):  lane l supplies A[l % 16][l / 16]
//   B (4x16):  lane l supplies B[l / 16][l % 16]
//   D (16x16): lane l holds D[l/16 + 4*r][l % 16] in element r = 0..3
// ---------------------------------------------------------------------------
template <int BM, int BN, int WAVES_M, int WAVES_N, bool A_ROWFAST = false, bool B_COLFAST = true>
struct MmaF64 {
  static constexpr int BK = 16;
  static constexpr int NT = 64 * WAVES_M * WAVES_N;
  static constexpr int WM = BM / WAVES_M;
  static constexpr int WN = BN / WAVES_N;
  static constexpr int TM = WM / 16;
  static constexpr int TN = WN / 16;
  static constexpr int LDA = BM + 2;
  static constexpr int LDB = BN + 2;
  static constexpr int LDS_DOUBLES = BK * (LDA + LDB);
  static constexpr int A_PER_T = (BM * BK) / NT;
  static constexpr int B_PER_T = (BK * BN) / NT;
  static_assert(WM % 16 == 0 && WN % 16 == 0, "wave tile must be a multiple of 16");
  static_assert((BM * BK) % NT == 0 && (BK * BN) % NT == 0, "tile not divisible by threads");

  f64x4 acc[TM][TN];
  int lane, wm, wn;

  __device__ __forceinline__ MmaF64() {
    lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    wm = wave / WAVES_N;
    wn = wave % WAVES_N;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
  }

  __device__ __forceinline__ static void a_coord(int e, int& r, int& kk) {
    if (A_ROWFAST) { r = e % BM; kk = e / BM; }
    else { r = e / BK; kk = e % BK; }
  }
  __device__ __forceinline__ static void b_coord(int e, int& kk, int& c) {
    if (B_COLFAST) { kk = e / BN; c = e % BN; }
    else { kk = e % BK; c = e / BK; }
  }

  // la(r, k): A element (tile-relative row r in [0,BM), absolute k); must return 0 out of range.
  // lb(k, c): B element (absolute k, tile-relative col c in [0,BN)).
  template <class LA, class LB>
  __device__ __forceinline__ void run(const LA& la, const LB& lb, int K, double* lds) {
    double* As = lds;
    double* Bs = lds + BK * LDA;
    const int tid = threadIdx.x;
    double ra[A_PER_T], rb[B_PER_T];
    auto fetch = [&](int k0) {
#pragma unroll
      for (int q = 0; q < A_PER_T; ++q) {
        int r, kk;
        a_coord(tid + q * NT, r, kk);
        ra[q] = la(r, k0 + kk);
      }
#pragma unroll
      for (int q = 0; q < B_PER_T; ++q) {
        int kk, c;
        b_coord(tid + q * NT, kk, c);
        rb[q] = lb(k0 + kk, c);
      }
    };
    const int nst = (K + BK - 1) / BK;
    if (nst > 0) fetch(0);
    for (int s = 0; s < nst; ++s) {
#pragma unroll
      for (int q = 0; q < A_PER_T; ++q) {
        int r, kk;
        a_coord(tid + q * NT, r, kk);
        As[kk * LDA + r] = ra[q];
      }
#pragma unroll
      for (int q = 0; q < B_PER_T; ++q) {
        int kk, c;
        b_coord(tid + q * NT, kk, c);
        Bs[kk * LDB + c] = rb[q];
      }
      __syncthreads();
      if (s + 1 < nst) fetch((s + 1) * BK);
#pragma unroll
      for (int k4 = 0; k4 < BK / 4; ++k4) {
        const int kr = k4 * 4 + (lane >> 4);
        double a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = As[kr * LDA + wm * WM + i * 16 + (lane & 15)];
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = Bs[kr * LDB + wn * WN + j * 16 + (lane & 15)];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
      }
      __syncthreads();
    }
  }

  // tile-relative coordinates of accumulator element acc[i][j][r]
  __device__ __forceinline__ int row(int i, int r) const { return wm * WM + i * 16 + (lane >> 4) + 4 * r; }
  __device__ __forceinline__ int col(int j) const { return wn * WN + j * 16 + (lane & 15); }

  template <class EP>
  __device__ __forceinline__ void store(const EP& ep) const {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) ep(row(i, r), col(j), acc[i][j][r]);
  }
};

// ---------------------------------------------------------------------------
// FP64 MFMA tile engine with per-thread operand pointers and a double-buffered
// LDS stage.  The loaders are evaluated once per tile: pa(r) is the start of A's
// row r (element k at pa(r)[k * sa]) and pb(c) the start of B's column c
// (element k at pb(c)[k * sb]); nullptr stands for a row or column of zeros.
// NT is a multiple of BM and of BN, so every thread stages one fixed row of A and
// one fixed column of B: a stage costs one load per element and no index
// arithmetic.  Stage s + 1 is loaded while stage s is multiplied and written to
// the other LDS buffer afterwards: one barrier per BK-deep stage.
// ---------------------------------------------------------------------------
template <int BM, int BN, int WAVES_M, int WAVES_N>
struct MmaF64P {
  static constexpr int BK = 16;
  static constexpr int NT = 64 * WAVES_M * WAVES_N;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  static constexpr int TM = WM / 16, TN = WN / 16;
  static constexpr int LDA = BM + 2, LDB = BN + 2;
  static constexpr int STAGE = BK * (LDA + LDB);
  static constexpr int LDS_DOUBLES = 2 * STAGE;
  static constexpr int A_PER_T = (BM * BK) / NT, B_PER_T = (BK * BN) / NT;
  static_assert(WM % 16 == 0 && WN % 16 == 0, "wave tile must be a multiple of 16");
  static_assert(NT % BM == 0 && NT % BN == 0, "every thread stages one row of A and one column of B");

  f64x4 acc[TM][TN];
  int lane, wm, wn;

  __device__ __forceinline__ MmaF64P() {
    lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    wm = wave / WAVES_N;
    wn = wave % WAVES_N;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
  }

  template <class PA, class PB>
  __device__ __forceinline__ void run(const PA& pa, const PB& pb, int64_t sa, int64_t sb, int K, double* lds) {
    const int tid = threadIdx.x;
    const int ra_row = tid % BM, ka0 = tid / BM;   // this thread's row of A, first k of its stage share
    const int rb_col = tid % BN, kb0 = tid / BN;
    const double* prow = pa(ra_row);
    const double* pcol = pb(rb_col);
    double ra[A_PER_T], rb[B_PER_T];
    auto fetch = [&](int k0) {
#pragma unroll
      for (int q = 0; q < A_PER_T; ++q) {
        const int k = k0 + ka0 + q * (NT / BM);
        ra[q] = 0.0;
        if (prow && k < K) ra[q] = prow[(int64_t)k * sa];
      }
#pragma unroll
      for (int q = 0; q < B_PER_T; ++q) {
        const int k = k0 + kb0 + q * (NT / BN);
        rb[q] = 0.0;
        if (pcol && k < K) rb[q] = pcol[(int64_t)k * sb];
      }
    };
    auto put = [&](int buf) {
      double* As = lds + buf * STAGE;
      double* Bs = As + BK * LDA;
#pragma unroll
      for (int q = 0; q < A_PER_T; ++q) As[(ka0 + q * (NT / BM)) * LDA + ra_row] = ra[q];
#pragma unroll
      for (int q = 0; q < B_PER_T; ++q) Bs[(kb0 + q * (NT / BN)) * LDB + rb_col] = rb[q];
    };
    const int nst = (K + BK - 1) / BK;
    if (nst > 0) {
      fetch(0);
      put(0);
    }
    __syncthreads();
    for (int s = 0; s < nst; ++s) {
      if (s + 1 < nst) fetch((s + 1) * BK);
      const double* As = lds + (s & 1) * STAGE;
      const double* Bs = As + BK * LDA;
#pragma unroll
      for (int k4 = 0; k4 < BK / 4; ++k4) {
        const int kr = k4 * 4 + (lane >> 4);
        double a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = As[kr * LDA + wm * WM + i * 16 + (lane & 15)];
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = Bs[kr * LDB + wn * WN + j * 16 + (lane & 15)];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
      }
      if (s + 1 < nst) put((s + 1) & 1);
      __syncthreads();
    }
  }

  __device__ __forceinline__ int row(int i, int r) const { return wm * WM + i * 16 + (lane >> 4) + 4 * r; }
  __device__ __forceinline__ int col(int j) const { return wn * WN + j * 16 + (lane & 15); }

  template <class EP>
  __device__ __forceinline__ void store(const EP& ep) const {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) ep(row(i, r), col(j), acc[i][j][r]);
  }
};

// ---------------------------------------------------------------------------
// BF16 MFMA tile engine with hi/lo split components.
//
// Both operands are K-contiguous in global memory and padded to a multiple of
// 8 bf16 along K: A as rows [m][k], B as columns [n][k] (i.e. B^T row-major).
// The loaders return, for a split component c and a tile-relative row/column,
// a pointer to that row's bf16 data (or nullptr: zero row).  A stage of BK=32
// is copied global -> registers -> LDS in 16-byte chunks, one stage ahead.
// With NA = NB = 2 (x = hi + lo) the engine accumulates in FP32
//     acc += A_hi B_hi + A_hi B_lo + A_lo B_hi      ("BF16x3")
// and with NA = NB = 1 the single product A_hi B_hi.
//
// v_mfma_f32_16x16x32_bf16 operand layout (one 64-lane wave):
//   A (16x32): lane l supplies A[l % 16][8*(l/16) + 0..7]
//   B (32x16): lane l supplies B[8*(l/16) + 0..7][l % 16]
//   D (16x16): lane l holds D[4*(l/16) + r][l % 16] in element r = 0..3
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16;

// round to nearest even: gfx950's v_cvt_pk_bf16_f32 (one instruction, where adding
// 0x7fff plus the lowest kept bit to the FP32 bits and truncating took three; the same
// result for every finite input)
__device__ __forceinline__ u16 f2bf_bits(float x) { return __builtin_bit_cast(u16, (__bf16)x); }
// two values in one instruction: a in the low half, b in the high half
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned f2bf2_bits(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2v){a, b}, bf16x2v));
}
__device__ __forceinline__ float bf_bits2f(u16 b) { return __uint_as_float(((unsigned)b) << 16); }
// four values split into packed pairs: hi = bf16(x), lo = bf16(x - hi), x[0] in the low
// half of hi.x
__device__ __forceinline__ void split4_bf16(const float (&x)[4], uint2& hi, uint2& lo) {
  hi.x = f2bf2_bits(x[0], x[1]);
  hi.y = f2bf2_bits(x[2], x[3]);
  lo.x = f2bf2_bits(x[0] - __uint_as_float(hi.x << 16), x[1] - __uint_as_float(hi.x & 0xffff0000u));
  lo.y = f2bf2_bits(x[2] - __uint_as_float(hi.y << 16), x[3] - __uint_as_float(hi.y & 0xffff0000u));
}
// x ~ hi + lo with hi = bf16(float(x)), lo = bf16(float(x - hi)): each rounded to FP32
// first, then to BF16.  (Without the empty register barriers the compiler merges the two
// conversions into one correctly rounded double -> BF16 conversion, which differs in the
// rare double-rounding cases and takes ten instructions instead of two.)
__device__ __forceinline__ void split_bf16(double x, u16& hi, u16& lo) {
  float f = (float)x;
  asm volatile("" : "+v"(f));
  hi = f2bf_bits(f);
  float g = (float)(x - (double)bf_bits2f(hi));
  asm volatile("" : "+v"(g));
  lo = f2bf_bits(g);
}

// DB: two LDS stage buffers (the next stage is written while the current one is read),
// one barrier per stage instead of two.  SB: a scheduling barrier between a K step's
// fragment reads and its MFMAs, so that all the reads are in flight before the first
// MFMA (the scheduler otherwise interleaves them and waits for LDS every few MFMAs).
template <int BM, int BN, int WAVES_M, int WAVES_N, int NA, int NB, int BK_ = 32, bool DB = false, bool SB = false>
struct MmaBF16 {
  static constexpr int BK = BK_;
  static constexpr int BM_ = BM, BN_ = BN;
  static constexpr int CPR = BK / 8;  // 16-byte chunks per row and stage
  static constexpr int LDK = BK + 8;  // bf16 per LDS row (keeps 16-B alignment)
  static constexpr int NT = 64 * WAVES_M * WAVES_N;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  static constexpr int TM = WM / 16, TN = WN / 16;
  static constexpr int A_CH = NA * BM * CPR;  // 16-byte chunks per stage
  static constexpr int B_CH = NB * BN * CPR;
  static constexpr int A_PER_T = (A_CH + NT - 1) / NT;
  static constexpr int B_PER_T = (B_CH + NT - 1) / NT;
  static constexpr int STAGE_U16 = (NA * BM + NB * BN) * LDK;
  static constexpr int LDS_BYTES = STAGE_U16 * 2 * (DB ? 2 : 1);
  static_assert(WM % 16 == 0 && WN % 16 == 0, "wave tile must be a multiple of 16");
  static_assert(BK % 32 == 0, "stage depth must be a multiple of the MFMA K (32)");

  f32x4 acc[TM][TN];
  int lane, wm, wn;

  __device__ __forceinline__ MmaBF16() {
    lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    wm = wave / WAVES_N;
    wn = wave % WAVES_N;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // pa(c, r) / pb(c, col): const u16* to the K-contiguous row of component c, or nullptr.
  // Kp: padded K (multiple of 8); rows hold at least Kp elements.  The loaders are
  // evaluated once per tile: each thread keeps the row pointers of the chunks it
  // moves and only advances k between stages.
  template <class PA, class PB>
  __device__ __forceinline__ void run(const PA& pa, const PB& pb, int Kp, void* ldsv) {
    u16* lds = reinterpret_cast<u16*>(ldsv);
    u16* As = lds;                    // [NA][BM][LDK]
    u16* Bs = lds + NA * BM * LDK;    // [NB][BN][LDK]
    const int tid = threadIdx.x;
    uint4 ra[A_PER_T], rb[B_PER_T];
    const u16* pA[A_PER_T];
    const u16* pB[B_PER_T];
    int oA[A_PER_T], oB[B_PER_T];   // LDS offsets of the chunks this thread stages
#pragma unroll
    for (int q = 0; q < A_PER_T; ++q) {
      const int e = tid + q * NT;
      pA[q] = nullptr;
      oA[q] = 0;
      if (e < A_CH) {
        const int ch = e % CPR, r = (e / CPR) % BM, c = (e / CPR) / BM;
        const u16* p = pa(c, r);
        if (p) pA[q] = p + ch * 8;
        oA[q] = (c * BM + r) * LDK + ch * 8;
      }
    }
#pragma unroll
    for (int q = 0; q < B_PER_T; ++q) {
      const int e = tid + q * NT;
      pB[q] = nullptr;
      oB[q] = 0;
      if (e < B_CH) {
        const int ch = e % CPR, r = (e / CPR) % BN, c = (e / CPR) / BN;
        const u16* p = pb(c, r);
        if (p) pB[q] = p + ch * 8;
        oB[q] = (c * BN + r) * LDK + ch * 8;
      }
    }
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    // (a branch, not "cond ? *p : zero": the select would load through a pointer to
    // the local zero, which moves the staging registers to scratch memory)
#define AFQ_BF16_FETCH(k0)                                                                     \
  {                                                                                            \
    _Pragma("unroll") for (int q = 0; q < A_PER_T; ++q) {                                      \
      const int k_ = (k0) + ((tid + q * NT) % CPR) * 8;                                        \
      ra[q] = zero;                                                                            \
      if (pA[q] && k_ < Kp) ra[q] = *reinterpret_cast<const uint4*>(pA[q] + (k0));             \
    }                                                                                          \
    _Pragma("unroll") for (int q = 0; q < B_PER_T; ++q) {                                      \
      const int k_ = (k0) + ((tid + q * NT) % CPR) * 8;                                        \
      rb[q] = zero;                                                                            \
      if (pB[q] && k_ < Kp) rb[q] = *reinterpret_cast<const uint4*>(pB[q] + (k0));             \
    }                                                                                          \
  }
    const int nst = (Kp + BK - 1) / BK;
    auto put = [&](int buf) {
      u16* base = lds + buf * STAGE_U16;
#pragma unroll
      for (int q = 0; q < A_PER_T; ++q)
        if (A_CH % NT == 0 || tid + q * NT < A_CH) *reinterpret_cast<uint4*>(base + oA[q]) = ra[q];
#pragma unroll
      for (int q = 0; q < B_PER_T; ++q)
        if (B_CH % NT == 0 || tid + q * NT < B_CH) *reinterpret_cast<uint4*>(base + NA * BM * LDK + oB[q]) = rb[q];
    };
    if (nst > 0) AFQ_BF16_FETCH(0)
    if (DB && nst > 0) {
      put(0);
      __syncthreads();
    }
    for (int s = 0; s < nst; ++s) {
      if (DB) {
        As = lds + (s & 1) * STAGE_U16;
        Bs = As + NA * BM * LDK;
      } else {
        put(0);
        __syncthreads();
      }
      if (s + 1 < nst) AFQ_BF16_FETCH((s + 1) * BK)
#pragma unroll
      for (int ks = 0; ks < BK / 32; ++ks) {
        const int koff = ks * 32 + 8 * (lane >> 4);
        bf16x8 a[NA][TM], b[NB][TN];
#pragma unroll
        for (int c = 0; c < NA; ++c)
#pragma unroll
          for (int i = 0; i < TM; ++i)
            a[c][i] = *reinterpret_cast<const bf16x8*>(As + (c * BM + wm * WM + i * 16 + (lane & 15)) * LDK + koff);
#pragma unroll
        for (int c = 0; c < NB; ++c)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            b[c][j] = *reinterpret_cast<const bf16x8*>(Bs + (c * BN + wn * WN + j * 16 + (lane & 15)) * LDK + koff);
        if constexpr (SB) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0][i], b[0][j], acc[i][j], 0, 0, 0);
            if (NB > 1) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0][i], b[NB - 1][j], acc[i][j], 0, 0, 0);
            if (NA > 1) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[NA - 1][i], b[0][j], acc[i][j], 0, 0, 0);
          }
      }
      if (DB && s + 1 < nst) put((s + 1) & 1);
      __syncthreads();
    }
#undef AFQ_BF16_FETCH
  }

  __device__ __forceinline__ int row(int i, int r) const { return wm * WM + i * 16 + 4 * (lane >> 4) + r; }
  __device__ __forceinline__ int col(int j) const { return wn * WN + j * 16 + (lane & 15); }

  template <class EP>
  __device__ __forceinline__ void store(const EP& ep) const {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) ep(row(i, r), col(j), acc[i][j][r]);
  }
};

// ---------------------------------------------------------------------------
// BF16 engine with element loaders: la(r, k) and lb(k, c) return floats that
// are rounded to bf16 when staged in LDS (the MLP's GEMMs, where operands come
// from FP32 master weights / activations in several layouts; the next stage's loads are in
// flight during this one's MFMAs, so the rounding waits for the write to LDS).  A_ROWFAST: consecutive
// threads load consecutive rows of A at one k (an operand that lies transposed in memory).
// ---------------------------------------------------------------------------
template <int BM, int BN, int WAVES_M, int WAVES_N, bool A_ROWFAST = false>
struct MmaBF16E {
  static constexpr int BK = 32;
  static constexpr int LDK = BK + 8;
  static constexpr int NT = 64 * WAVES_M * WAVES_N;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  static constexpr int TM = WM / 16, TN = WN / 16;
  static constexpr int A_PER_T = BM * BK / NT, B_PER_T = BK * BN / NT;
  static constexpr int LDS_BYTES = (BM + BN) * LDK * 2;
  static_assert((BM * BK) % NT == 0 && (BK * BN) % NT == 0, "tile not divisible by threads");
  f32x4 acc[TM][TN];
  int lane, wm, wn;
  __device__ __forceinline__ MmaBF16E() {
    lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    wm = wave / WAVES_N;
    wn = wave % WAVES_N;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  template <class LA, class LB>
  __device__ __forceinline__ void run(const LA& la, const LB& lb, int K, void* ldsv) {
    u16* As = reinterpret_cast<u16*>(ldsv);
    u16* Bs = As + BM * LDK;
    const int tid = threadIdx.x;
    float ra[A_PER_T], rb[B_PER_T];
    auto fetch = [&](int k0) {
#pragma unroll
      for (int q = 0; q < A_PER_T; ++q) {
        const int e = tid + q * NT, r = A_ROWFAST ? e % BM : e / BK, kk = A_ROWFAST ? e / BM : e % BK;
        ra[q] = la(r, k0 + kk);
      }
#pragma unroll
      for (int q = 0; q < B_PER_T; ++q) {
        const int e = tid + q * NT, kk = e / BN, c = e % BN;
        rb[q] = lb(k0 + kk, c);
      }
    };
    const int nst = (K + BK - 1) / BK;
    if (nst > 0) fetch(0);
    for (int s = 0; s < nst; ++s) {
#pragma unroll
      for (int q = 0; q < A_PER_T; ++q) {
        const int e = tid + q * NT, r = A_ROWFAST ? e % BM : e / BK, kk = A_ROWFAST ? e / BM : e % BK;
        As[r * LDK + kk] = f2bf_bits(ra[q]);
      }
#pragma unroll
      for (int q = 0; q < B_PER_T; ++q) {
        const int e = tid + q * NT, kk = e / BN, c = e % BN;
        Bs[c * LDK + kk] = f2bf_bits(rb[q]);
      }
      __syncthreads();
      if (s + 1 < nst) fetch((s + 1) * BK);
      const int koff = 8 * (lane >> 4);
      bf16x8 a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        a[i] = *reinterpret_cast<const bf16x8*>(As + (wm * WM + i * 16 + (lane & 15)) * LDK + koff);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        b[j] = *reinterpret_cast<const bf16x8*>(Bs + (wn * WN + j * 16 + (lane & 15)) * LDK + koff);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
      __syncthreads();
    }
  }
  __device__ __forceinline__ int row(int i, int r) const { return wm * WM + i * 16 + 4 * (lane >> 4) + r; }
  __device__ __forceinline__ int col(int j) const { return wn * WN + j * 16 + (lane & 15); }
  template <class EP>
  __device__ __forceinline__ void store(const EP& ep) const {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) ep(row(i, r), col(j), acc[i][j][r]);
  }
};

}  // namespace afq
