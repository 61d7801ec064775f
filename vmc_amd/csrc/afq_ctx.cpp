// Host side of the C ABI (include/vmc_afqmc.h): the device context that holds
// one rank's walker population, its setup math (mean-field shifts, one-body
// propagator) and the stream-ordered step.  The step's arithmetic runs in the
// HIP kernels of afq_kernels.hip; nothing here falls back to the CPU.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <numeric>
#include <random>
#include <complex>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

#include "afq_group.hpp"
#include "afq_internal.hpp"

using afq::DevState;

namespace {

thread_local std::string g_create_error;

struct DevError : std::runtime_error {
  int code;
  DevError(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

void hip_check(hipError_t e, const char* what) {
  if (e != hipSuccess)
    throw DevError(AFQ_ERR_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
}
void launch_check(const char* what) { hip_check(hipGetLastError(), what); }

template <class T>
T* dalloc(size_t n) {
  void* p = nullptr;
  if (n == 0) n = 1;
  hip_check(hipMalloc(&p, n * sizeof(T)), "hipMalloc");
  return static_cast<T*>(p);
}

// exp(s*H) for a real symmetric H by scaling and squaring of the Taylor series
// (the reference uses Eigen's Pade MatrixBase::exp, DQMC/DQMCWalker.cpp:102).
std::vector<double> expm_scaled(const std::vector<double>& H, int N, double s) {
  double nrm = 0.0;
  for (int i = 0; i < N; ++i) {
    double r = 0.0;
    for (int j = 0; j < N; ++j) r += std::fabs(H[(size_t)i * N + j]);
    nrm = std::max(nrm, r);
  }
  nrm *= std::fabs(s);
  int sq = 0;
  while (nrm > 0.125) { nrm *= 0.5; ++sq; }
  const double a = s / std::ldexp(1.0, sq);
  std::vector<double> X((size_t)N * N), term((size_t)N * N), tmp((size_t)N * N), E((size_t)N * N, 0.0);
  for (size_t q = 0; q < X.size(); ++q) X[q] = a * H[q];
  for (int i = 0; i < N; ++i) E[(size_t)i * N + i] = 1.0;
  term = E;
  auto matmul = [&](const std::vector<double>& A, const std::vector<double>& B, std::vector<double>& C) {
    std::fill(C.begin(), C.end(), 0.0);
    for (int i = 0; i < N; ++i)
      for (int k = 0; k < N; ++k) {
        const double aik = A[(size_t)i * N + k];
        if (aik == 0.0) continue;
        const double* b = &B[(size_t)k * N];
        double* c = &C[(size_t)i * N];
        for (int j = 0; j < N; ++j) c[j] += aik * b[j];
      }
  };
  for (int k = 1; k <= 18; ++k) {  // ||X|| <= 1/8: 18 terms reach far below double rounding
    matmul(term, X, tmp);
    for (size_t q = 0; q < tmp.size(); ++q) { term[q] = tmp[q] / k; E[q] += term[q]; }
  }
  for (int k = 0; k < sq; ++k) {
    matmul(E, E, tmp);
    E.swap(tmp);
  }
  return E;
}

}  // namespace


hipEvent_t afq_ctx::ev_get() {
  hipEvent_t e;
  if (!pool.empty()) {
    e = pool.back();
    pool.pop_back();
    return e;
  }
  hip_check(hipEventCreateWithFlags(&e, hipEventDisableSystemFence), "hipEventCreate");
  return e;
}
void afq_ctx::stage_begin(int st, EvPair& p) {
  if (!timing) return;
  if (pending.size() > 4096) resolve();
  p.a = ev_get();
  p.first = true;
  p.stage = st;
  hip_check(hipEventRecord(p.a, stream), "hipEventRecord");
}
// A marker costs the stream a packet that waits for the work before it, so where nothing lies
// between two stages one marker ends the first and begins the second.  Only its time stamp is
// read, so it flushes no caches (no system fence).  A block of five steps at N = 10, 128 walkers:
// two markers a stage 1123 us, shared ones 893, without the fence 794.
void afq_ctx::stage_next(int st, EvPair& p) {
  if (!timing) return;
  stage_end(p);
  p.a = p.b;
  p.first = false;
  p.stage = st;
}
void afq_ctx::stage_end(EvPair& p) {
  if (!timing) return;
  p.b = ev_get();
  hip_check(hipEventRecord(p.b, stream), "hipEventRecord");
  pending.push_back(p);
}
void afq_ctx::resolve() {
  for (auto& p : pending) {
    hip_check(hipEventSynchronize(p.b), "hipEventSynchronize");
    float ms = 0.f;
    hip_check(hipEventElapsedTime(&ms, p.a, p.b), "hipEventElapsedTime");
    stage_ms[p.stage] += ms;
    if (p.first) pool.push_back(p.a);   // a later pair's a is its predecessor's b
    pool.push_back(p.b);
  }
  pending.clear();
}

namespace {

int fail(afq_ctx* c, int code, const std::string& m) {
  if (c) c->err = m;
  else g_create_error = m;
  return code;
}

#define AFQ_GUARD_BEGIN try {
#define AFQ_GUARD_END(ctx)                                      \
  }                                                             \
  catch (const DevError& e) { return fail(ctx, e.code, e.what()); } \
  catch (const std::exception& e) { return fail(ctx, AFQ_ERR_ARG, e.what()); }

struct Stage {
  afq_ctx* c;
  afq_ctx::EvPair p;
  Stage(afq_ctx* c_, int st) : c(c_) { c->stage_begin(st, p); }
  void next(int st) { c->stage_next(st, p); }   // where nothing is launched between the two stages
  ~Stage() { try { c->stage_end(p); } catch (...) {} }
};

void free_all(DevState& s) {
  double* ptrs[] = {s.E2, s.Lp2, s.P2, s.E, s.Lp, s.R, s.phi[0], s.phi[1], s.hphi[0], s.hphi[1], s.mf, s.psi, s.theta, s.fb,
                    s.logO, s.e1, s.logdet, s.weights, s.factors, s.psi2, s.theta2, s.fb2, s.logO2, s.e12,
                    s.fields, s.sft, s.P, s.t0, s.t1, s.accb, s.draws, s.Xp, s.eloc, s.ho, s.cum, s.Sg, s.stats};
  for (double* p : ptrs)
    if (p) (void)hipFree(p);
  if (s.idx) (void)hipFree(s.idx);
  if (s.live) (void)hipFree(s.live);
  if (s.gfresh) (void)hipFree(s.gfresh);
  if (s.nlive) (void)hipFree(s.nlive);
  if (s.vhs_blk) (void)hipFree(s.vhs_blk);
  if (s.ncap) (void)hipFree(s.ncap);
  unsigned short* hp[] = {s.Rb_hi, s.Rb_lo, s.Rf, s.Rf_lo, s.Tb_hi, s.Tb_lo, s.Lt_hi, s.Lt_lo, s.Fb_hi, s.Fb_lo,
                          s.Vh, s.Vl, s.Ub[0], s.Ub[1], s.Ub[2], s.Dh, s.Dl};
  for (unsigned short* p : hp)
    if (p) (void)hipFree(p);
  void* vp[] = {s.Rq8, s.Tq8, s.rinv8, s.tinv8, s.fbp};
  for (void* p : vp)
    if (p) (void)hipFree(p);
}

// bf16 operand copies for the low-precision exchange (allocated on first use)
void ensure_lowprec(DevState& s, hipStream_t st) {
  if (s.Rb_hi) return;
  int64_t rows = 0;
  for (int q = 0; q < s.nslots; ++q) rows += (int64_t)s.G * s.slot[q].n;
  s.Rb_hi = dalloc<unsigned short>(rows * s.Np);
  s.Rb_lo = dalloc<unsigned short>(rows * s.Np);
  s.Tb_hi = dalloc<unsigned short>((int64_t)s.W * s.ctot * s.Np);
  s.Tb_lo = dalloc<unsigned short>((int64_t)s.W * s.ctot * s.Np);
  if (s.nslots == 2) {
    s.fbp_rows = 2 * s.W;
    s.fbp = dalloc<float>(2 * (int64_t)s.fbp_rows * s.G);
  }
  afq::launch_rsplit(s, st);
  launch_check("rsplit");
  if (const int64_t nf = afq::rfrag_elems(s, s.rf_off)) {
    s.Rf = dalloc<unsigned short>(nf);
    s.Rf_lo = dalloc<unsigned short>(nf);
    afq::launch_rfrag(s, st);
    launch_check("rfrag");
  }
}

// bf16 operand copies for the low-precision VHS (allocated on first use)
void ensure_vhs_lowprec(DevState& s, hipStream_t st) {
  if (s.Lt_hi) return;
  s.Gp = (s.G + 7) / 8 * 8;
  s.Lt_hi = dalloc<unsigned short>(s.T * s.Gp);
  s.Lt_lo = dalloc<unsigned short>(s.T * s.Gp);
  s.Fb_hi = dalloc<unsigned short>((int64_t)s.W * 2 * s.Gp);
  s.Fb_lo = dalloc<unsigned short>((int64_t)s.W * 2 * s.Gp);
  std::vector<int> blk;
  for (int i0 = 0; i0 < s.N; i0 += 16)
    for (int j0 = 0; j0 < s.N && j0 <= i0 + 15; j0 += 8) {
      blk.push_back(i0);
      blk.push_back(j0);
    }
  s.nvhs_blk = (int)blk.size() / 2;
  s.vhs_blk = dalloc<int>(blk.size());
  hip_check(hipMemcpyAsync(s.vhs_blk, blk.data(), blk.size() * sizeof(int), hipMemcpyHostToDevice, st), "H2D");
  hip_check(hipStreamSynchronize(st), "sync");
  afq::launch_lt_split(s, st);
  launch_check("lt_split");
}

// split-BF16 Taylor operands (allocated on first use), zero so that the orbital pads
// of every chunk stay zero
void ensure_prop_lowprec(DevState& s, hipStream_t st) {
  if (s.Vh) return;
  s.Nq = (s.N + 15) / 16 * 16;
  const int ncolc = s.det_n[0] + (s.ndets_prop > 1 ? s.det_n[1] : 0);
  const int64_t nv = (int64_t)s.W * s.Nq * s.N * 2;       // u16 per V plane (chunks x N x 32)
  const int64_t nu = (int64_t)s.W * 4 * ncolc * s.Nq;     // u16 per u buffer
  s.Vh = dalloc<unsigned short>(nv);
  s.Vl = dalloc<unsigned short>(nv);
  for (int k = 0; k < 3; ++k) s.Ub[k] = dalloc<unsigned short>(nu);
  afq::launch_fill(reinterpret_cast<double*>(s.Vh), nv / 4, 0.0, st);
  afq::launch_fill(reinterpret_cast<double*>(s.Vl), nv / 4, 0.0, st);
  for (int k = 0; k < 3; ++k) afq::launch_fill(reinterpret_cast<double*>(s.Ub[k]), nu / 4, 0.0, st);
  const int64_t nd = (int64_t)s.N * afq::onebody_pitch(s.N);
  s.Dh = dalloc<unsigned short>(nd);
  s.Dl = dalloc<unsigned short>(nd);
  afq::launch_d_split(s, st);   // again at every afq_prep_prop
  launch_check("prop split buffers");
}

// force bias of the current theta in the context's force-bias precision
void run_force_bias(const DevState& s, hipStream_t st) {
  if (s.prec_fb == AFQ_PREC_FP64) afq::launch_force_bias(s, st);
  else afq::launch_force_bias_lp(s, s.prec_fb, st);
}

bool exchange_prec_ok(int p) {
  return p == AFQ_PREC_FP64 || p == AFQ_PREC_BF16X3 || p == AFQ_PREC_BF16;
}
// the exchange contraction also runs in e4m3
bool exchange_only_prec_ok(int p) { return exchange_prec_ok(p) || p == AFQ_PREC_FP8; }

// e4m3 exchange operands (allocated on first use; the rotated Cholesky is converted once)
void ensure_q8(DevState& s, hipStream_t st) {
  if (s.Rq8) return;
  s.Npq = (s.N + 15) / 16 * 16;
  int64_t rows = 0;
  for (int q = 0; q < s.nslots; ++q) rows += (int64_t)s.G * s.slot[q].n;
  s.Rq8 = dalloc<unsigned char>(rows * s.Npq);
  s.rinv8 = dalloc<float>(s.G);
  s.Tq8 = dalloc<unsigned char>((int64_t)s.W * s.ctot * s.Npq);
  s.tinv8 = dalloc<float>(2 * (int64_t)s.W);
  afq::launch_rq8(s, st);
  launch_check("rq8");
}
// operand buffers of an exchange precision
void ensure_exchange_prec(DevState& s, int prec, hipStream_t st) {
  if (prec == AFQ_PREC_FP8) ensure_q8(s, st);
  else if (prec != AFQ_PREC_FP64) ensure_lowprec(s, st);
}

// Walker-dependent buffers for a population of W.
void alloc_walkers(DevState& s) {
  const int64_t W = s.W;
  s.psi = dalloc<double>(2 * W * s.ms);
  s.psi2 = dalloc<double>(2 * W * s.ms);
  s.theta = dalloc<double>(2 * W * s.Ktot);
  s.theta2 = dalloc<double>(2 * W * s.Ktot);
  s.fb = dalloc<double>(2 * W * s.G);
  s.fb2 = dalloc<double>(2 * W * s.G);
  s.logO = dalloc<double>(2 * W);
  s.logO2 = dalloc<double>(2 * W);
  s.e1 = dalloc<double>(2 * W * s.nslots);
  s.e12 = dalloc<double>(2 * W * s.nslots);
  s.logdet = dalloc<double>(2 * W * s.nslots);
  s.weights = dalloc<double>(W);
  s.factors = dalloc<double>(W);
  s.fields = dalloc<double>(2 * W * s.G);
  s.sft = dalloc<double>(4 * W);
  s.P = dalloc<double>(2 * W * (int64_t)s.N * s.N);
  s.t0 = dalloc<double>(2 * W * s.ms);
  s.t1 = dalloc<double>(2 * W * s.ms);
  s.accb = dalloc<double>(2 * W * s.ms);
  s.draws = dalloc<double>(W * s.G);
  s.Xp = dalloc<double>(2 * (int64_t)s.nslots * W * s.ngt_cap);
  s.Sg = dalloc<double>((int64_t)W * s.nslots * 64 * 128);
  const bool big = W * s.nslots * 64 * 128 >= 2 * W * s.Ktot;
  s.fbw = big ? s.Sg : s.theta2;
  s.fbw_doubles = big ? W * s.nslots * 64 * 128 : 2 * W * s.Ktot;
  s.eloc = dalloc<double>(W);
  s.ho = dalloc<double>(4 * W);
  s.cum = dalloc<double>(W);
  s.idx = dalloc<int>(W);
  s.live = dalloc<int>(W);
  s.gfresh = dalloc<int>(W);
  s.nlive = dalloc<int>(1);
  s.ncap = dalloc<unsigned long long>(2);
  s.stats = dalloc<double>(afq::STATS_DOUBLES);
}

void upload(double* d, const double* h, size_t n, hipStream_t st) {
  hip_check(hipMemcpyAsync(d, h, n * sizeof(double), hipMemcpyHostToDevice, st), "hipMemcpyAsync H2D");
}
void download(double* h, const double* d, size_t n, hipStream_t st) {
  hip_check(hipMemcpyAsync(h, d, n * sizeof(double), hipMemcpyDeviceToHost, st), "hipMemcpyAsync D2H");
  hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
}

// Small results to the host: one kernel a result writes them to pinned memory, then one
// synchronization for all.  hipMemcpyAsync to the caller's pageable memory and a synchronization
// for each took, on a block of five steps at N = 10, 128 walkers (14 results), 794 us, now 617.  Larger
// results, which the bus bounds, are copied directly.
struct Result {
  void* h;
  const void* d;
  size_t n;   // 8-byte words
};
constexpr size_t PIN_WORDS = 32768, TMP_KEEP = size_t(64) << 20;
void readback(afq_ctx* c, std::initializer_list<Result> results) {
  size_t tot = 0;
  for (const Result& r : results)
    if (r.h) tot += r.n;
  if (tot > PIN_WORDS) {
    for (const Result& r : results)
      if (r.h) download(static_cast<double*>(r.h), static_cast<const double*>(r.d), r.n, c->stream);
    return;
  }
  if (tot == 0) return;
  std::lock_guard<std::mutex> lk(c->pin_mu);
  if (!c->pin) hip_check(hipHostMalloc(reinterpret_cast<void**>(&c->pin), PIN_WORDS * sizeof(double), hipHostMallocDefault), "hipHostMalloc");
  size_t o = 0;
  for (const Result& r : results) {
    if (!r.h) continue;
    afq::launch_copy_small(static_cast<const double*>(r.d), c->pin + o, (int)r.n, c->stream);
    o += r.n;
  }
  launch_check("readback");
  hip_check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
  o = 0;
  for (const Result& r : results) {
    if (!r.h) continue;
    std::memcpy(r.h, c->pin + o, r.n * sizeof(double));
    o += r.n;
  }
}

// Mean-field shifts and propagator constant of DQMCWalker::prepPropR
// (DQMC/DQMCWalker.cpp:32-103), phaseless branch; returns h1' = h1Mod - sum mf_g (i L_g).
// With unrestricted integrals (prepPropU, :106-187) the shifts sum both spins' terms
// and h1p2 receives the down-spin h1'.
void prep_math(afq_ctx* c, const double* gref_up, const double* gref_dn, double dt,
               std::vector<double>& mf, std::vector<double>& h1p, double& pc, std::vector<double>* h1p2 = nullptr) {
  DevState& s = c->s;
  const int N = s.N, G = s.G;
  const size_t NN = (size_t)N * N;
  h1p = c->h1mod;
  if (s.uints && h1p2) *h1p2 = c->h1modd;
  mf.assign(2 * (size_t)G, 0.0);
  double constant = -s.ecore;  // ene0 cancels in the phaseless constant
  auto rd = [&](double l) { return s.ref_compat ? (double)(float)l : l; };
  for (int g = 0; g < G; ++g) {
    const double* L = &c->chol[g * NN];
    const double* Ld = s.uints ? &c->chold[g * NN] : nullptr;
    double a = 0.0;
    if (s.uints)
      for (size_t q = 0; q < NN; ++q) a += gref_up[q] * rd(L[q]) + gref_dn[q] * rd(Ld[q]);
    else
      for (size_t q = 0; q < NN; ++q) a += (gref_up[q] + gref_dn[q]) * rd(L[q]);
    // mf = i a;  constant -= mf^2/2 = +a^2/2;  h1' -= mf * (i L) = + a L
    mf[2 * g] = 0.0;
    mf[2 * g + 1] = a;
    constant += 0.5 * a * a;
    for (size_t q = 0; q < NN; ++q) h1p[q] += a * rd(L[q]);
    if (s.uints && h1p2)
      for (size_t q = 0; q < NN; ++q) (*h1p2)[q] += a * rd(Ld[q]);
  }
  pc = constant;
  (void)dt;
}

void green_ref(const double* ref, int N, int n, std::vector<double>& G) {
  // G = ref (ref^T ref)^-1 ref^T by Gauss-Jordan on the n x n Gram matrix
  std::vector<double> S((size_t)n * n, 0.0), inv((size_t)n * n, 0.0);
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) {
      double a = 0.0;
      for (int k = 0; k < N; ++k) a += ref[(size_t)k * n + i] * ref[(size_t)k * n + j];
      S[(size_t)i * n + j] = a;
    }
  for (int i = 0; i < n; ++i) inv[(size_t)i * n + i] = 1.0;
  for (int k = 0; k < n; ++k) {
    int p = k;
    for (int i = k + 1; i < n; ++i)
      if (std::fabs(S[(size_t)i * n + k]) > std::fabs(S[(size_t)p * n + k])) p = i;
    for (int j = 0; j < n; ++j) {
      std::swap(S[(size_t)k * n + j], S[(size_t)p * n + j]);
      std::swap(inv[(size_t)k * n + j], inv[(size_t)p * n + j]);
    }
    const double d = S[(size_t)k * n + k];
    for (int j = 0; j < n; ++j) { S[(size_t)k * n + j] /= d; inv[(size_t)k * n + j] /= d; }
    for (int i = 0; i < n; ++i) {
      if (i == k) continue;
      const double f = S[(size_t)i * n + k];
      for (int j = 0; j < n; ++j) {
        S[(size_t)i * n + j] -= f * S[(size_t)k * n + j];
        inv[(size_t)i * n + j] -= f * inv[(size_t)k * n + j];
      }
    }
  }
  G.assign((size_t)N * N, 0.0);
  std::vector<double> tmp((size_t)N * n, 0.0);  // ref * inv
  for (int i = 0; i < N; ++i)
    for (int j = 0; j < n; ++j) {
      double a = 0.0;
      for (int k = 0; k < n; ++k) a += ref[(size_t)i * n + k] * inv[(size_t)k * n + j];
      tmp[(size_t)i * n + j] = a;
    }
  for (int i = 0; i < N; ++i)
    for (int j = 0; j < N; ++j) {
      double a = 0.0;
      for (int k = 0; k < n; ++k) a += tmp[(size_t)i * n + k] * ref[(size_t)j * n + k];
      G[(size_t)i * N + j] = a;
    }
}

// Green's function, log overlap and force bias of the current population.
void refresh_walkers(afq_ctx* c, bool overlaps_from_dets) {
  DevState& s = c->s;
  {
    Stage t(c, afq::ST_GREEN);
    afq::launch_green(s, true, c->stream);
    launch_check("green");
  }
  s.theta_stale = false;
  if (overlaps_from_dets) {
    afq::launch_logO_from_logdet(s, c->stream);
    launch_check("logO");
  }
  Stage t(c, afq::ST_FB);
  run_force_bias(s, c->stream);
  launch_check("force_bias");
}

// theta of every walker after an eager comb (which does not carry it) or new weights,
// for the entry points that read it before the next propagation; the force bias of the
// walkers of nonzero weight with it (a step computes it only for the walkers it leaves
// alive, and new weights may revive others)
void ensure_theta(afq_ctx* c) {
  DevState& s = c->s;
  if (!s.theta_stale) return;
  Stage t(c, afq::ST_GREEN);
  afq::launch_green(s, true, c->stream);
  launch_check("green");
  t.next(afq::ST_FB);
  run_force_bias(s, c->stream);
  launch_check("force_bias");
  s.theta_stale = false;
  c->fb_stale = false;
}

void free_cv(afq_ctx* c) {
  afq::RiskSort& r = c->rsort;
  for (void* p : {(void*)c->cvS, (void*)c->cvEK, (void*)c->cvEJ, (void*)c->cvPinv, (void*)c->cvSel, (void*)c->cvX,
                  (void*)c->cvD, (void*)c->cvCenter, (void*)c->cvNsel, (void*)c->cvTame, (void*)c->cvRisky,
                  (void*)r.kin, (void*)r.kout, (void*)r.iin, (void*)r.iout, r.tmp})
    if (p) (void)hipFree(p);
  c->cvS = c->cvEK = c->cvEJ = c->cvD = c->cvCenter = nullptr;
  c->cvPinv = nullptr;
  c->cvSel = c->cvNsel = c->cvTame = nullptr;
  c->cvRisky = nullptr;
  c->cvX = nullptr;
  c->rsort = afq::RiskSort();
  c->cv_halfw = 0.0;
}

// buffers of the control variate (both surrogate kinds)
void ensure_cv(afq_ctx* c) {
  DevState& s = c->s;
  if (!c->cvS) c->cvS = dalloc<double>(s.W);
  if (!c->cvEK) c->cvEK = dalloc<double>(s.W);
  if (!c->cvEJ) c->cvEJ = dalloc<double>(s.W);
  if (!c->cvPinv) c->cvPinv = dalloc<float>(s.W);
  if (!c->cvD) c->cvD = dalloc<double>(s.W);
  if (!c->cvSel) c->cvSel = dalloc<int>(s.W);
  if (!c->cvNsel) c->cvNsel = dalloc<int>(1);
  if (!c->cvTame) c->cvTame = dalloc<int>(s.W);
  if (!c->cvRisky) c->cvRisky = dalloc<unsigned char>(s.W);
}

// the risk stratum of the live walkers into c->cvRisky (E_J in c->cvEJ), on the device
void risk_split_dev(afq_ctx* c) {
  DevState& s = c->s;
  afq::RiskSort& r = c->rsort;
  if (!r.kin) {
    r.kin = dalloc<double>(s.W);
    r.kout = dalloc<double>(s.W);
    r.iin = dalloc<int>(s.W);
    r.iout = dalloc<int>(s.W);
    r.tmp_bytes = afq::risk_sort_bytes(s.W);
    r.tmp = dalloc<unsigned char>(r.tmp_bytes);
  }
  afq::launch_risk_split(s, c->cvEJ, c->cv_risk, r, c->cvRisky, c->stream);
  launch_check("risk split");
}

void free_mlp(afq_ctx* c) {
  afq::Mlp& m = c->mlp;
  std::vector<void*> ptrs = {m.mu, m.sd, m.lossbuf, m.ws, m.xn, m.X, m.Y, c->cvX};
  for (int l = 0; l < 4; ++l)
    for (void* p : {(void*)m.w[l], (void*)m.b[l], (void*)m.mw[l], (void*)m.vw[l], (void*)m.mb[l], (void*)m.vb[l],
                    (void*)m.gw[l], (void*)m.gb[l], (void*)m.z[l], (void*)m.h[l], (void*)m.dh[l]})
      ptrs.push_back(p);
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  m = afq::Mlp();
  c->cvX = nullptr;
}

// synchronous copy ordered after all work queued on the context's (non-blocking) stream
hipError_t scopy(afq_ctx* c, void* dst, const void* src, size_t bytes, hipMemcpyKind kind) {
  hipError_t e = hipStreamSynchronize(c->stream);
  if (e != hipSuccess) return e;
  e = hipMemcpyAsync(dst, src, bytes, kind, c->stream);
  if (e != hipSuccess) return e;
  return hipStreamSynchronize(c->stream);
}

int64_t mlp_nparams(const afq::Mlp& m) {
  int64_t n = 0;
  for (int l = 0; l < 4; ++l) n += (int64_t)m.dims[l] * m.dims[l + 1] + m.dims[l + 1];
  return n;
}

}  // namespace

// Driver support: keep a context's last error readable after the context is gone, and
// set the message of a failure the driver itself detects.
__attribute__((visibility("hidden"))) void afq_keep_error(const afq_ctx* c, int rc) {
  if (c && rc != AFQ_OK) g_create_error = c->err;
}
__attribute__((visibility("hidden"))) void afq_set_error(afq_ctx* c, const char* msg) {
  if (c) c->err = msg;
}

extern "C" {

int afq_version(void) { return AFQ_ABI_VERSION; }

const char* afq_last_error(const afq_ctx* ctx) {
  return ctx ? ctx->err.c_str() : g_create_error.c_str();
}

int afq_create(const afq_ham* ham, const afq_trial* left, const afq_params* params, afq_ctx** out) {
  if (!ham || !left || !params || !out) return fail(nullptr, AFQ_ERR_ARG, "null argument");
  *out = nullptr;
  const int N = ham->norb, na = ham->nalpha, nb = ham->nbeta, G = ham->nchol, W = params->nwalk;
  if (N <= 0 || na <= 0 || nb < 0 || G <= 0 || W <= 0 || na > N || nb > N)
    return fail(nullptr, AFQ_ERR_ARG, "bad sizes");
  if (!ham->h1 || !ham->h1_mod || !ham->chol || !left->phi_up || (!left->rhf && !left->phi_dn))
    return fail(nullptr, AFQ_ERR_ARG, "null Hamiltonian / trial pointer");
  if ((params->walker_rhf || left->rhf) && na != nb)
    return fail(nullptr, AFQ_ERR_ARG, "RHF walker / RHF trial needs nalpha == nbeta");
  if (nb == 0) return fail(nullptr, AFQ_ERR_UNSUPPORTED, "nbeta == 0 not supported");
  if (na > 64 || nb > 64)
    return fail(nullptr, AFQ_ERR_UNSUPPORTED, "more than 64 electrons per spin not supported by this build");
  if (!exchange_prec_ok(params->prec_fb) || !exchange_prec_ok(params->prec_vhs) ||
      !exchange_only_prec_ok(params->prec_exchange))
    return fail(nullptr, AFQ_ERR_UNSUPPORTED, "requested precision mode not available");
  if (params->ref_compat && params->prec_vhs != AFQ_PREC_FP64)
    return fail(nullptr, AFQ_ERR_UNSUPPORTED, "ref_compat rounds the VHS itself; it needs prec_vhs = FP64");
  const bool uints = ham->h1_dn || ham->h1_mod_dn || ham->chol_dn;
  if (uints && !(ham->h1_dn && ham->h1_mod_dn && ham->chol_dn))
    return fail(nullptr, AFQ_ERR_ARG, "unrestricted integrals need h1_dn, h1_mod_dn and chol_dn");
  if (uints && (params->walker_rhf || left->rhf))
    return fail(nullptr, AFQ_ERR_UNSUPPORTED, "unrestricted integrals need a UHF trial and UHF walkers");
  if (uints && params->prec_vhs != AFQ_PREC_FP64)
    return fail(nullptr, AFQ_ERR_UNSUPPORTED, "unrestricted integrals need the FP64 VHS");
  afq_ctx* c = new afq_ctx();
  try {
    c->params = *params;
    hip_check(hipSetDevice(params->device), "hipSetDevice");
    hip_check(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking), "hipStreamCreate");
    DevState& s = c->s;
    s.N = N; s.na = na; s.nb = nb; s.G = G; s.GE = G; s.W = W;
    s.T = (int64_t)N * (N + 1) / 2;
    s.ms = (int64_t)N * (na + nb);
    s.walker_rhf = params->walker_rhf != 0;
    s.trial_rhf = left->rhf != 0;
    s.ref_compat = params->ref_compat != 0;
    s.uints = uints;
    s.ecore = ham->ecore;
    s.weight_cap = params->weight_cap > 0 ? params->weight_cap : std::max(100.0, W / 10.0);
    s.det_n[0] = na; s.det_n[1] = nb;
    s.det_off[0] = 0; s.det_off[1] = (int64_t)N * na;
    s.ndets_prop = s.walker_rhf ? 1 : 2;
    if (s.walker_rhf && s.trial_rhf) {
      s.nslots = 1;
      s.slot[0] = afq::Slot{na, 0, 0, 2, 0};
      s.slot[1] = s.slot[0];
    } else {
      s.nslots = 2;
      s.slot[0] = afq::Slot{na, 0, 0, 1, 0};
      s.slot[1] = afq::Slot{nb, s.walker_rhf ? 0 : 1, s.trial_rhf ? 0 : 1, 1, (int64_t)N * na};
    }
    s.Ktot = 0;
    for (int q = 0; q < s.nslots; ++q) s.Ktot += (int64_t)N * s.slot[q].n;
    s.fbo = afq::fb_order(G, s.Ktot, s.nslots);
    s.Np = (N + 7) / 8 * 8;
    s.ctot = 0;
    for (int q = 0; q < s.nslots; ++q) s.ctot += 2 * s.slot[q].n;
    s.prec_exchange = params->prec_exchange;
    s.prec_fb = params->prec_fb;
    s.prec_vhs = params->prec_vhs;
    int ngt = 0;
    for (int q = 0; q < s.nslots; ++q)
      ngt = std::max(ngt, (G + afq::exchange_tile_g(s.slot[q].n) - 1) / afq::exchange_tile_g(s.slot[q].n));
    s.ngt_cap = ngt;
    // host copies for setup math
    const size_t NN = (size_t)N * N;
    c->h1.assign(ham->h1, ham->h1 + NN);
    c->h1mod.assign(ham->h1_mod, ham->h1_mod + NN);
    c->chol.assign(ham->chol, ham->chol + (size_t)G * NN);
    if (uints) {
      c->h1d.assign(ham->h1_dn, ham->h1_dn + NN);
      c->h1modd.assign(ham->h1_mod_dn, ham->h1_mod_dn + NN);
      c->chold.assign(ham->chol_dn, ham->chol_dn + (size_t)G * NN);
    }
    c->phi[0].assign(left->phi_up, left->phi_up + (size_t)N * na);
    c->phi[1] = left->rhf ? c->phi[0] : std::vector<double>(left->phi_dn, left->phi_dn + (size_t)N * nb);
    // device Hamiltonian / trial
    double* Ld = dalloc<double>((size_t)G * NN);
    upload(Ld, c->chol.data(), (size_t)G * NN, c->stream);
    s.Lp = dalloc<double>((size_t)G * s.T + 1);   // pairs of columns are read at any offset
    afq::launch_pack_chol(Ld, s.Lp, N, G, s.T, s.ref_compat, c->stream);
    launch_check("pack_chol");
    double* Ldd = nullptr;  // down-spin vectors (unrestricted integrals)
    if (uints) {
      Ldd = dalloc<double>((size_t)G * NN);
      upload(Ldd, c->chold.data(), (size_t)G * NN, c->stream);
      s.Lp2 = dalloc<double>((size_t)G * s.T + 1);
      afq::launch_pack_chol(Ldd, s.Lp2, N, G, s.T, s.ref_compat, c->stream);
      launch_check("pack_chol");
    }
    s.R = dalloc<double>((size_t)G * s.Ktot);
    for (int p = 0; p < 2; ++p) {
      const int n = p == 0 ? na : nb;
      s.phi[p] = dalloc<double>((size_t)N * n);
      upload(s.phi[p], c->phi[p].data(), (size_t)N * n, c->stream);
      std::vector<double> hp((size_t)N * n, 0.0);
      const std::vector<double>& h1s = (uints && p == 1) ? c->h1d : c->h1;  // spin p's h1
      for (int i = 0; i < N; ++i)
        for (int k = 0; k < N; ++k) {
          const double h = h1s[(size_t)i * N + k];
          for (int j = 0; j < n; ++j) hp[(size_t)i * n + j] += h * c->phi[p][(size_t)k * n + j];
        }
      s.hphi[p] = dalloc<double>((size_t)N * n);
      upload(s.hphi[p], hp.data(), hp.size(), c->stream);
    }
    for (int q = 0; q < s.nslots; ++q) {
      const afq::Slot& sl = s.slot[q];
      // unrestricted integrals: each spin's rows from its own vectors (DQMC/Hamiltonian.cpp:99-107)
      afq::launch_rotate_chol((uints && sl.phi == 1) ? Ldd : Ld, s.phi[sl.phi], s.R, N, sl.n, G, s.Ktot, sl.koff,
                              c->stream);
      launch_check("rotate_chol");
    }
    hip_check(hipStreamSynchronize(c->stream), "setup sync");
    hip_check(hipFree(Ld), "hipFree");
    if (Ldd) hip_check(hipFree(Ldd), "hipFree");
    s.E = dalloc<double>(NN);
    if (uints) {
      s.E2 = dalloc<double>(NN);
      s.P2 = dalloc<double>(2 * (size_t)W * NN);
    }
    s.mf = dalloc<double>(2 * (size_t)G);
    alloc_walkers(s);
    afq::launch_fill(s.weights, W, 0.0, c->stream);
    afq::launch_fill(s.stats, afq::STATS_DOUBLES, 0.0, c->stream);
    ensure_exchange_prec(s, s.prec_exchange, c->stream);
    if (s.prec_fb != AFQ_PREC_FP64) ensure_lowprec(s, c->stream);
    if (s.prec_vhs != AFQ_PREC_FP64) ensure_vhs_lowprec(s, c->stream);
    hip_check(hipStreamSynchronize(c->stream), "setup sync");
  } catch (const DevError& e) {
    free_all(c->s);
    delete c;
    return fail(nullptr, e.code, e.what());
  } catch (const std::exception& e) {
    free_all(c->s);
    delete c;
    return fail(nullptr, AFQ_ERR_DEVICE, e.what());
  }
  *out = c;
  return AFQ_OK;
}

int afq_destroy(afq_ctx* c) {
  if (!c) return AFQ_OK;
  (void)hipStreamSynchronize(c->stream);
  for (auto& p : c->pending) {
    if (p.first) (void)hipEventDestroy(p.a);
    (void)hipEventDestroy(p.b);
  }
  for (hipEvent_t e : c->pool) (void)hipEventDestroy(e);
  free_all(c->s);
  free_mlp(c);
  free_cv(c);
  if (c->rdmAcc) (void)hipFree(c->rdmAcc);
  if (c->rdmPart) (void)hipFree(c->rdmPart);
  if (c->tmp) (void)hipFree(c->tmp);
  if (c->pin) (void)hipHostFree(c->pin);
  (void)hipStreamDestroy(c->stream);
  delete c;
  return AFQ_OK;
}

int afq_set_precision(afq_ctx* c, int32_t prec_fb, int32_t prec_vhs, int32_t prec_exchange) {
  if (!c) return AFQ_ERR_ARG;
  if (!exchange_prec_ok(prec_fb) || !exchange_prec_ok(prec_vhs) || !exchange_only_prec_ok(prec_exchange))
    return fail(c, AFQ_ERR_UNSUPPORTED, "requested precision mode not available");
  if (c->s.ref_compat && prec_vhs != AFQ_PREC_FP64)
    return fail(c, AFQ_ERR_UNSUPPORTED, "ref_compat rounds the VHS itself; it needs prec_vhs = FP64");
  if (c->s.uints && prec_vhs != AFQ_PREC_FP64)
    return fail(c, AFQ_ERR_UNSUPPORTED, "unrestricted integrals need the FP64 VHS");
  AFQ_GUARD_BEGIN
  ensure_exchange_prec(c->s, prec_exchange, c->stream);
  if (prec_fb != AFQ_PREC_FP64) ensure_lowprec(c->s, c->stream);
  if (prec_vhs != AFQ_PREC_FP64) ensure_vhs_lowprec(c->s, c->stream);
  c->s.prec_exchange = prec_exchange;
  c->s.prec_fb = prec_fb;
  c->s.prec_vhs = prec_vhs;
  c->params.prec_exchange = prec_exchange;
  c->params.prec_fb = prec_fb;
  c->params.prec_vhs = prec_vhs;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_set_prop_precision(afq_ctx* c, int32_t prec_prop) {
  if (!c) return AFQ_ERR_ARG;
  if (prec_prop != AFQ_PREC_FP64 && prec_prop != AFQ_PREC_BF16X3)
    return fail(c, AFQ_ERR_UNSUPPORTED, "propagation precision must be FP64 or BF16X3");
  if (prec_prop != AFQ_PREC_FP64 && c->s.ref_compat)
    return fail(c, AFQ_ERR_UNSUPPORTED, "ref_compat needs the FP64 propagation");
  if (prec_prop != AFQ_PREC_FP64 && c->s.uints)
    return fail(c, AFQ_ERR_UNSUPPORTED, "unrestricted integrals need the FP64 propagation");
  AFQ_GUARD_BEGIN
  if (prec_prop != AFQ_PREC_FP64) ensure_prop_lowprec(c->s, c->stream);
  c->s.prec_prop = prec_prop;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_set_nchol_ene(afq_ctx* c, int32_t n) {
  if (!c) return AFQ_ERR_ARG;
  if (n < 0 || n > c->s.G) return fail(c, AFQ_ERR_ARG, "nchol_ene out of range");
  c->s.GE = n;
  return AFQ_OK;
}

int afq_prep_prop(afq_ctx* c, const double* ref_up, const double* ref_dn, const double* rdm_up,
                  const double* rdm_dn, double dt, double ene0) {
  if (!c) return AFQ_ERR_ARG;
  (void)ene0;
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  if (!(dt > 0.0)) return fail(c, AFQ_ERR_ARG, "dt must be positive");
  std::vector<double> gu, gd;
  if (rdm_up && rdm_dn) {
    gu.assign(rdm_up, rdm_up + (size_t)s.N * s.N);
    gd.assign(rdm_dn, rdm_dn + (size_t)s.N * s.N);
  } else {
    if (!ref_up || !ref_dn) return fail(c, AFQ_ERR_ARG, "reference determinant required");
    green_ref(ref_up, s.N, s.na, gu);
    green_ref(ref_dn, s.N, s.nb, gd);
  }
  std::vector<double> mf, h1p, h1p2;
  double pc = 0.0;
  prep_math(c, gu.data(), gd.data(), dt, mf, h1p, pc, &h1p2);
  const std::vector<double> E = expm_scaled(h1p, s.N, -dt / 2.0);
  s.dt = dt;
  s.prop_const_re = pc;
  s.prop_const_im = 0.0;
  upload(s.mf, mf.data(), mf.size(), c->stream);
  upload(s.E, E.data(), E.size(), c->stream);
  if (s.uints) {
    const std::vector<double> E2 = expm_scaled(h1p2, s.N, -dt / 2.0);
    upload(s.E2, E2.data(), E2.size(), c->stream);
  }
  if (s.Dh) afq::launch_d_split(s, c->stream);
  hip_check(hipStreamSynchronize(c->stream), "prep sync");
  c->prepped = true;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_set_walkers(afq_ctx* c, const double* dets, const double* overlaps, const double* weights) {
  if (!c || !dets) return c ? fail(c, AFQ_ERR_ARG, "null dets") : AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  upload(s.psi, dets, 2 * (size_t)s.W * s.ms, c->stream);
  if (weights) upload(s.weights, weights, s.W, c->stream);
  else afq::launch_fill(s.weights, s.W, 1.0, c->stream);
  if (overlaps) {
    std::vector<double> lo(2 * (size_t)s.W);
    for (int w = 0; w < s.W; ++w) {
      const std::complex<double> o(overlaps[2 * w], overlaps[2 * w + 1]);
      lo[2 * w] = std::log(std::abs(o));
      lo[2 * w + 1] = std::arg(o);
    }
    upload(s.logO, lo.data(), lo.size(), c->stream);
  }
  refresh_walkers(c, overlaps == nullptr);
  hip_check(hipStreamSynchronize(c->stream), "set_walkers sync");
  c->have_walkers = true;
  c->fb_stale = false;
  c->last_measure_clipped = false;
  c->last_exact_all = false;   // the last measurement's per-walker partials were of other walkers
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_get_walkers(afq_ctx* c, double* dets, double* overlaps, double* weights) {
  if (!c) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  if (dets) {
    download(dets, s.psi, 2 * (size_t)s.W * s.ms, c->stream);
    if (s.walker_rhf) {  // det[1] mirrors det[0] for an RHF walker (DQMC/DQMCWalker.cpp:486)
      const size_t n0 = 2 * (size_t)s.N * s.na;
      for (int w = 0; w < s.W; ++w)
        std::memcpy(dets + 2 * (size_t)w * s.ms + 2 * s.det_off[1], dets + 2 * (size_t)w * s.ms, n0 * sizeof(double));
    }
  }
  if (overlaps) {
    std::vector<double> lo(2 * (size_t)s.W);
    readback(c, {{lo.data(), s.logO, lo.size()}});
    for (int w = 0; w < s.W; ++w) {
      const std::complex<double> o = std::exp(std::complex<double>(lo[2 * w], lo[2 * w + 1]));
      overlaps[2 * w] = o.real();
      overlaps[2 * w + 1] = o.imag();
    }
  }
  if (weights) readback(c, {{weights, s.weights, (size_t)s.W}});
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_get_weights(afq_ctx* c, double* weights) { return afq_get_walkers(c, nullptr, nullptr, weights); }

int afq_set_weights(afq_ctx* c, const double* weights) {
  if (!c || !weights) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  upload(c->s.weights, weights, c->s.W, c->stream);
  c->s.tb_live = false;
  c->s.tb_post = false;
  // a walker of weight zero may carry a theta older than its orbitals (a step skips the
  // theta of walkers it kills); new weights can make it live again, so the next reader
  // recomputes theta for every walker
  c->s.theta_stale = true;
  c->fb_stale = true;
  c->last_exact_all = false;   // the exchange partials of revived walkers are not current
  hip_check(hipStreamSynchronize(c->stream), "sync");
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_propagate(afq_ctx* c, const double* draws, uint64_t seed, uint64_t step, double eshift,
                  double* factors, int64_t* n_capped) {
  if (!c) return AFQ_ERR_ARG;
  if (!c->prepped || !c->have_walkers) return fail(c, AFQ_ERR_STATE, "afq_prep_prop and afq_set_walkers first");
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  // walkers revived by afq_set_weights get theta and the force bias of their current
  // orbitals before the fields read the force bias
  if (c->fb_stale) ensure_theta(c);
  c->last_exact_all = false;
  if (draws) upload(s.draws, draws, (size_t)s.W * s.G, c->stream);
  {
    Stage t(c, afq::ST_FIELDS);
    afq::launch_fields(s, draws ? s.draws : nullptr, seed, step, c->stream);
    launch_check("fields");
    t.next(afq::ST_VHS);
    if (s.prec_vhs == AFQ_PREC_FP64) afq::launch_vhs(s, c->stream);
    else afq::launch_vhs_lp(s, s.prec_vhs, c->stream);
    launch_check("vhs");
    const bool one = afq::prop_in_one(s);
    if (!one) {
      t.next(afq::ST_PROP);
      afq::launch_expmul_pre(s, c->stream);
    }
    t.next(afq::ST_TAYLOR);
    afq::launch_taylor(s, c->stream);
    if (!one) {
      t.next(afq::ST_PROP);
      afq::launch_expmul_post(s, c->stream);
    }
    launch_check("propagate");
    t.next(afq::ST_GREEN);
    // after a comb every walker's overlap matrix is recomputed, propagated or not
    afq::launch_green_pre(s, s.theta_stale, c->stream);
    launch_check("green");
    t.next(afq::ST_WEIGHT);
    afq::launch_weight(s, eshift, true, c->stream);
    launch_check("weight");
    t.next(afq::ST_GREEN);
    afq::launch_theta_post(s, c->stream);   // theta of the walkers still alive
    launch_check("theta");
    s.theta_stale = false;
    t.next(afq::ST_FB);
    run_force_bias(s, c->stream);
    launch_check("force_bias");
  }
  afq::launch_step_stats(s, c->stream);   // sum of the weights, live and propagated counts
  launch_check("step stats");
  c->last_measure_clipped = false;
  unsigned long long capped = 0;
  readback(c, {{factors, s.factors, (size_t)s.W}, {n_capped ? &capped : nullptr, s.ncap, 1}});
  if (n_capped) *n_capped = (int64_t)capped;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_orthogonalize(afq_ctx* c) {
  if (!c) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  Stage t(c, afq::ST_ORTHO);
  afq::launch_qr(c->s, c->stream);
  launch_check("qr");
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

// Two-level control variate, on the device.  The surrogate predicts y = E_K - E_J on
// every walker; the exact exchange is evaluated on (a) every walker of the risk stratum
// (the fraction cv_risk of the live walkers whose Coulomb energy E_J lies farthest from
// the median; inclusion probability 1) and (b) one walker drawn uniformly from each
// consecutive block of cv_minv remaining live walkers (inclusion probability 1/b for a
// block of b).  The Horvitz-Thompson correction keeps every walker's estimate unbiased
// for its exact local energy.  Nothing comes back to the host unless a fallback
// threshold is set: then the residual RMS of the sample is read, and every walker is
// evaluated exactly instead when it exceeds the threshold.
static int measure_cv(afq_ctx* c, double delta, double* eloc) {
  DevState& s = c->s;
  afq::Mlp& m = c->mlp;
  const hipStream_t st = c->stream;
  if (c->cv_kind == AFQ_SURR_MLP && !m.ready) return fail(c, AFQ_ERR_STATE, "surrogate not trained");
  ensure_cv(c);
  afq::launch_live_list(s, st);
  if (c->cv_kind == AFQ_SURR_MLP) {
    afq::launch_features(s, nullptr, s.W, c->cvX, 0, st);
    afq::launch_predict(s, m, c->cvX, s.W, c->cvS, st);
    afq::launch_ej(s, c->cvEJ, st);
  } else {
    // reduced-precision exchange of every live walker: S = E_K(reduced) - E_J
    if (s.GE > 0) {
      Stage t(c, afq::ST_EXLP);
      afq::launch_exchange_lp(s, s.live, s.W, c->cv_prec, st, s.nlive);
      launch_check("exchange (surrogate level)");
    }
    afq::launch_ek(s, s.live, s.W, c->cvS, nullptr, 0, st, s.nlive);
    afq::launch_ej(s, c->cvEJ, st);
    afq::launch_sub(c->cvS, c->cvEJ, s.W, st);
  }
  launch_check("surrogate level");
  const unsigned char* risky = nullptr;
  int nrisk_max = 0;
  if (c->cv_risk > 0.0) {
    risk_split_dev(c);
    risky = c->cvRisky;
    nrisk_max = std::min(s.W, (int)std::ceil(c->cv_risk * s.W));
  }
  afq::launch_cv_select(s, risky, c->cv_minv, c->cv_seed, c->cv_draw++, c->cv_force, c->cvTame, c->cvSel, c->cvNsel,
                        c->cvPinv, st);
  launch_check("cv select");
  // the exact set: at most the risk stratum plus one walker per block
  const int bound = std::min(s.W, nrisk_max + (s.W + c->cv_minv - 1) / c->cv_minv);
  if (s.GE > 0) {
    Stage t(c, afq::ST_ENERGY);
    if (s.prec_exchange == AFQ_PREC_FP64) afq::launch_exchange(s, c->cvSel, bound, st, c->cvNsel);
    else afq::launch_exchange_lp(s, c->cvSel, bound, s.prec_exchange, st, c->cvNsel);
    launch_check("exchange (subset)");
  }
  afq::launch_ek(s, c->cvSel, bound, c->cvEK, nullptr, 0, st, c->cvNsel);
  const bool clip = c->cv_halfw > 0.0 && c->cvCenter;
  afq::launch_energy_cv(s, c->cvS, c->cvEK, c->cvPinv, delta, s.stats + afq::SS_CVOFF, clip ? c->cvCenter : nullptr,
                        c->cv_nwr, c->cv_halfw, c->cvD, st);
  afq::launch_cv_stats(s, c->cvS, c->cvEK, c->cvEJ, c->cvD, c->cvPinv, c->cvSel, c->cvNsel, st);
  launch_check("energy_cv");
  bool fallback = false;
  if (c->cv_fallback > 0.0) {
    double rms = 0.0;
    download(&rms, s.stats + afq::SS_CVRMS, 1, st);
    if (rms > c->cv_fallback) {
      fallback = true;
      if (s.GE > 0) {
        Stage t(c, afq::ST_ENERGY);
        if (s.prec_exchange == AFQ_PREC_FP64) afq::launch_exchange(s, s.live, s.W, st, s.nlive);
        else afq::launch_exchange_lp(s, s.live, s.W, s.prec_exchange, st, s.nlive);
      }
      afq::launch_energy(s, nullptr, s.W, delta, st);
      launch_check("fallback exact");
    }
  }
  if (!fallback) afq::launch_cv_offset(s, c->cv_offset_rate, st);
  c->cv_last_fallback = fallback;
  c->cv_nfallback += fallback ? 1 : 0;
  c->last_exact_all = fallback;
  c->last_measure_clipped = !fallback && clip;
  if (eloc) readback(c, {{eloc, s.eloc, (size_t)s.W}});
  return AFQ_OK;
}

int afq_measure(afq_ctx* c, int32_t mode, double delta, double* eloc, double* ham_ovlp) {
  if (!c) return AFQ_ERR_ARG;
  if (mode != AFQ_ENERGY_EXACT && mode != AFQ_ENERGY_SURROGATE)
    return fail(c, AFQ_ERR_UNSUPPORTED, "energy mode not available");
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  ensure_theta(c);
  if (mode == AFQ_ENERGY_SURROGATE) {
    if (ham_ovlp) return fail(c, AFQ_ERR_ARG, "ham_ovlp is not produced by the surrogate mode");
    return measure_cv(c, delta, eloc);
  }
  // the walkers of nonzero weight, listed on the device (the grid covers all W and the
  // exchange tiles past the list's length exit)
  afq::launch_live_list(s, c->stream);
  if (s.GE > 0) {
    Stage t(c, afq::ST_ENERGY);  // the exchange contraction alone
    if (s.prec_exchange == AFQ_PREC_FP64) afq::launch_exchange(s, s.live, s.W, c->stream, s.nlive);
    else afq::launch_exchange_lp(s, s.live, s.W, s.prec_exchange, c->stream, s.nlive);
    launch_check("exchange");
  }
  afq::launch_energy(s, nullptr, s.W, delta, c->stream);
  launch_check("energy");
  c->last_exact_all = true;
  c->last_measure_clipped = false;
  readback(c, {{eloc, s.eloc, (size_t)s.W}, {ham_ovlp, s.ho, 4 * (size_t)s.W}});
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_ham_and_overlap(afq_ctx* c, const double* dets, int32_t ndet, int32_t nchol_ene, double* out) {
  if (!c || !dets || !out || ndet <= 0) return c ? fail(c, AFQ_ERR_ARG, "bad arguments") : AFQ_ERR_ARG;
  if (nchol_ene < 0 || nchol_ene > c->s.G) return fail(c, AFQ_ERR_ARG, "nchol_ene out of range");
  AFQ_GUARD_BEGIN
  // a temporary population of ndet walkers sharing the Hamiltonian buffers, in one block that the
  // context keeps up to TMP_KEEP (calls on one context take turns with it)
  std::lock_guard<std::mutex> lk(c->tmp_mu);
  DevState t = afq::temporary_population(c->s, ndet, nchol_ene);
  afq::Carve size{nullptr};
  afq::carve_population(t, ndet, size);
  if (size.off > c->tmp_bytes) {
    if (c->tmp) (void)hipFree(c->tmp);
    c->tmp = nullptr;
    c->tmp_bytes = 0;
    c->tmp = dalloc<unsigned char>(size.off);
    c->tmp_bytes = size.off;
  }
  afq::Carve cv{c->tmp};
  afq::carve_population(t, ndet, cv);
  struct GiveBack {
    afq_ctx* c;
    ~GiveBack() {
      if (c->tmp_bytes <= TMP_KEEP) return;
      (void)hipFree(c->tmp);
      c->tmp = nullptr;
      c->tmp_bytes = 0;
    }
  } give_back{c};
  upload(t.psi, dets, 2 * (size_t)ndet * t.ms, c->stream);
  afq::launch_temporary(t, c->stream);
  launch_check("ham_and_overlap");
  readback(c, {{out, t.ho, 4 * (size_t)ndet}});
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_force_bias(afq_ctx* c, double* fb) {
  if (!c || !fb) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  if (c->fb_stale) ensure_theta(c);
  download(fb, c->s.fb, 2 * (size_t)c->s.W * c->s.G, c->stream);
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_overlap(afq_ctx* c, double* overlaps) { return afq_get_walkers(c, nullptr, overlaps, nullptr); }

int afq_comb(afq_ctx* c, double zeta, double* total_weight) {
  if (!c) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  {
    Stage t(c, afq::ST_COMB);
    afq::launch_comb(c->s, zeta, c->stream);
    launch_check("comb");
  }
  c->last_exact_all = false;  // the last measurement's per-walker partials refer to the old walkers
  if (total_weight) readback(c, {{total_weight, c->s.cum + (c->s.W - 1), 1}});
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

// Mixed-estimator one-body density matrix (DQMC/MixedEstimator.cpp:492-510).
int afq_rdm_reset(afq_ctx* c) {
  if (!c) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  if (!c->rdmAcc) c->rdmAcc = dalloc<double>(s.Ktot + 1);
  afq::launch_fill(c->rdmAcc, s.Ktot + 1, 0.0, c->stream);
  launch_check("rdm reset");
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_rdm_accumulate(afq_ctx* c) {
  if (!c) return AFQ_ERR_ARG;
  if (!c->have_walkers) return fail(c, AFQ_ERR_STATE, "afq_set_walkers first");
  if (!c->rdmAcc) {
    const int rc = afq_rdm_reset(c);
    if (rc) return rc;
  }
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  if (!c->rdmPart) c->rdmPart = dalloc<double>(afq::rdm_part_doubles(s));
  ensure_theta(c);
  afq::launch_rdm_accumulate(s, c->rdmPart, c->rdmAcc, c->stream);
  launch_check("rdm accumulate");
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

// RDM_s(i, j) = sum_e Phi_s(i, e) acc_s(j, e) / sum w: the running average of
// Re(theta_s Phi_s^T)^T.  spin_summed: the slots' matrices added with their
// multiplicity (RHF::oneRDM, DQMC/RHF.cpp:64-67); otherwise [up | down]
// (UHF::oneRDM, DQMC/UHF.cpp:68-72): slot 0 is the up spin and slot 1 the down
// spin, and a single slot of multiplicity 2 stands for both.
int afq_get_one_rdm(afq_ctx* c, int32_t spin_summed, double* rdm, double* cumulative_weight) {
  if (!c || !rdm) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  const int N = s.N;
  const size_t NN = (size_t)N * N;
  std::fill(rdm, rdm + (spin_summed ? 1 : 2) * NN, 0.0);
  std::vector<double> acc(s.Ktot + 1, 0.0);
  if (c->rdmAcc) download(acc.data(), c->rdmAcc, s.Ktot + 1, c->stream);
  const double cw = acc[s.Ktot];
  if (cumulative_weight) *cumulative_weight = cw;
  if (cw == 0.0) return AFQ_OK;
  std::vector<double> M(NN);
  for (int q = 0; q < s.nslots; ++q) {
    const afq::Slot& sl = s.slot[q];
    const double* ph = c->phi[sl.phi].data();  // N x n_s row-major
    const double* a = acc.data() + sl.koff;    // [j][e]: orbital j, electron e
    for (int i = 0; i < N; ++i)
      for (int j = 0; j < N; ++j) {
        double v = 0.0;
        for (int e = 0; e < sl.n; ++e) v += ph[(size_t)i * sl.n + e] * a[(size_t)j * sl.n + e];
        M[(size_t)i * N + j] = v / cw;
      }
    if (spin_summed) {
      for (size_t k = 0; k < NN; ++k) rdm[k] += sl.mult * M[k];
    } else {
      for (int d = 0; d < 2; ++d)
        if (q == d || sl.mult == 2)
          for (size_t k = 0; k < NN; ++k) rdm[d * NN + k] += M[k];
    }
  }
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_stage_times(afq_ctx* c, double* ms10, int32_t reset) {
  static_assert(afq::ST_COUNT == AFQ_NSTAGES, "stage count");
  if (!c) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  c->resolve();
  for (int i = 0; i < afq::ST_COUNT; ++i) {
    if (ms10) ms10[i] = c->stage_ms[i];
    if (reset) c->stage_ms[i] = 0.0;
  }
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_debug_gemm_f64(const double* A, const double* B, double* C, int32_t M, int32_t N, int32_t K) {
  if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0) return fail(nullptr, AFQ_ERR_ARG, "bad gemm arguments");
  try {
    double* dA = dalloc<double>((size_t)M * K);
    double* dB = dalloc<double>((size_t)K * N);
    double* dC = dalloc<double>((size_t)M * N);
    upload(dA, A, (size_t)M * K, nullptr);
    upload(dB, B, (size_t)K * N, nullptr);
    afq::launch_debug_gemm(dA, dB, dC, M, N, K, nullptr);
    launch_check("debug_gemm");
    download(C, dC, (size_t)M * N, nullptr);
    (void)hipFree(dA); (void)hipFree(dB); (void)hipFree(dC);
  } catch (const DevError& e) {
    return fail(nullptr, e.code, e.what());
  }
  return AFQ_OK;
}

int afq_debug_gemm_bf16(const double* A, const double* B, float* C, int32_t M, int32_t N, int32_t K,
                        int32_t passes) {
  if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0 || (passes != 1 && passes != 3))
    return fail(nullptr, AFQ_ERR_ARG, "bad gemm arguments");
  try {
    const int64_t Kp = (K + 7) / 8 * 8;
    double* dA = dalloc<double>((size_t)M * K);
    double* dB = dalloc<double>((size_t)K * N);
    float* dC = dalloc<float>((size_t)M * N);
    void* scr = dalloc<uint16_t>((size_t)2 * (M + N) * Kp);
    upload(dA, A, (size_t)M * K, nullptr);
    upload(dB, B, (size_t)K * N, nullptr);
    afq::launch_debug_gemm_bf16(dA, dB, dC, M, N, K, passes, scr, nullptr);
    launch_check("debug_gemm_bf16");
    hip_check(hipMemcpy(C, dC, (size_t)M * N * sizeof(float), hipMemcpyDeviceToHost), "D2H");
    (void)hipFree(dA); (void)hipFree(dB); (void)hipFree(dC); (void)hipFree(scr);
  } catch (const DevError& e) {
    return fail(nullptr, e.code, e.what());
  }
  return AFQ_OK;
}

int afq_debug_copy(int64_t bytes) {
  if (bytes <= 0) return fail(nullptr, AFQ_ERR_ARG, "bad size");
  try {
    const int64_t n = bytes / 8;
    double* a = dalloc<double>(n);
    double* b = dalloc<double>(n);
    afq::launch_fill(a, n, 1.0, nullptr);
    afq::launch_copy_calib(a, b, n, nullptr);
    launch_check("copy_calib");
    hip_check(hipDeviceSynchronize(), "sync");
    (void)hipFree(a); (void)hipFree(b);
  } catch (const DevError& e) {
    return fail(nullptr, e.code, e.what());
  }
  return AFQ_OK;
}

// ------------------------------------------------------------------ surrogate
int afq_surrogate_init(afq_ctx* c, int32_t hidden, uint64_t seed, int64_t capacity) {
  if (!c || hidden <= 0 || capacity < 0) return c ? fail(c, AFQ_ERR_ARG, "bad surrogate arguments") : AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  free_mlp(c);
  DevState& s = c->s;
  afq::Mlp& m = c->mlp;
  const int F = s.G + 2 * s.N;
  m.dims[0] = F; m.dims[1] = hidden; m.dims[2] = hidden; m.dims[3] = hidden; m.dims[4] = 1;
  m.Bcap = std::max(s.W, 4096);
  std::mt19937_64 rng(seed);
  for (int l = 0; l < 4; ++l) {
    const int64_t nw = (int64_t)m.dims[l] * m.dims[l + 1], nb = m.dims[l + 1];
    std::vector<float> wi(nw), bi(nb, 0.f);
    // uniform(-a, a), a = sqrt(6 / (fan_in + fan_out))
    const double a = std::sqrt(6.0 / (m.dims[l] + m.dims[l + 1]));
    std::uniform_real_distribution<double> U(-a, a);
    for (auto& x : wi) x = (float)U(rng);
    float** bufs[] = {&m.w[l], &m.mw[l], &m.vw[l], &m.gw[l]};
    for (float** b : bufs) *b = dalloc<float>(nw);
    float** bbufs[] = {&m.b[l], &m.mb[l], &m.vb[l], &m.gb[l]};
    for (float** b : bbufs) *b = dalloc<float>(nb);
    hip_check(scopy(c, m.w[l], wi.data(), nw * 4, hipMemcpyHostToDevice), "H2D");
    hip_check(scopy(c, m.b[l], bi.data(), nb * 4, hipMemcpyHostToDevice), "H2D");
    std::vector<float> zw(nw, 0.f), zb(nb, 0.f);
    hip_check(scopy(c, m.mw[l], zw.data(), nw * 4, hipMemcpyHostToDevice), "H2D");
    hip_check(scopy(c, m.vw[l], zw.data(), nw * 4, hipMemcpyHostToDevice), "H2D");
    hip_check(scopy(c, m.mb[l], zb.data(), nb * 4, hipMemcpyHostToDevice), "H2D");
    hip_check(scopy(c, m.vb[l], zb.data(), nb * 4, hipMemcpyHostToDevice), "H2D");
    m.z[l] = dalloc<float>((int64_t)m.Bcap * m.dims[l + 1]);
    m.h[l] = dalloc<float>((int64_t)m.Bcap * m.dims[l + 1]);
    m.dh[l] = dalloc<float>((int64_t)m.Bcap * m.dims[l + 1]);
  }
  m.mu = dalloc<float>(F);
  m.sd = dalloc<float>(F);
  std::vector<float> z0(F, 0.f), o1(F, 1.f);
  hip_check(scopy(c, m.mu, z0.data(), F * 4, hipMemcpyHostToDevice), "H2D");
  hip_check(scopy(c, m.sd, o1.data(), F * 4, hipMemcpyHostToDevice), "H2D");
  m.lossbuf = dalloc<float>(1);
  m.xn = dalloc<float>((int64_t)m.Bcap * F);
  m.ws = dalloc<float>(afq::mlp_ws_floats(m.dims, m.Bcap));
  m.cap = capacity;
  if (capacity > 0) {
    m.X = dalloc<float>(capacity * F);
    m.Y = dalloc<float>(capacity);
  }
  ensure_cv(c);
  c->cvX = dalloc<float>((int64_t)s.W * F);
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_surrogate_collect(afq_ctx* c, int64_t* total) {
  if (!c || !c->mlp.dims[0]) return c ? fail(c, AFQ_ERR_STATE, "surrogate not initialised") : AFQ_ERR_ARG;
  if (!c->last_exact_all) return fail(c, AFQ_ERR_STATE, "collect needs an exact measurement of every walker");
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  afq::Mlp& m = c->mlp;
  ensure_theta(c);
  ensure_cv(c);
  // the risk stratum is always evaluated exactly, so the surrogate learns the rest: the
  // live walkers outside it, in walker order (the draw with blocks of one walker lists
  // them after the stratum)
  afq::launch_live_list(s, c->stream);
  const unsigned char* risky = nullptr;
  if (c->cv_risk > 0.0) {
    afq::launch_ej(s, c->cvEJ, c->stream);
    risk_split_dev(c);
    risky = c->cvRisky;
  }
  afq::launch_cv_select(s, risky, 1, 0, 0, 0, c->cvTame, c->cvSel, c->cvNsel, c->cvPinv, c->stream);
  launch_check("collect list");
  double cnt[2];
  download(cnt, s.stats + afq::SS_NRISK, 2, c->stream);   // SS_NRISK, SS_NRAND
  const int nrisk = (int)cnt[0], ntame = (int)cnt[1];
  const int64_t room = m.cap - m.n;
  const int nadd = (int)std::min<int64_t>(room, (int64_t)ntame);
  if (nadd > 0) {
    afq::launch_features(s, c->cvSel + nrisk, nadd, m.X, m.n, c->stream);
    afq::launch_ek(s, c->cvSel + nrisk, nadd, nullptr, m.Y, m.n, c->stream);
    launch_check("collect");
    hip_check(hipStreamSynchronize(c->stream), "sync");
    m.n += nadd;
  }
  if (total) *total = m.n;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_surrogate_load(afq_ctx* c, const float* X, const float* Y, int64_t n, int64_t* total) {
  if (!c || !X || !Y || n < 0) return c ? fail(c, AFQ_ERR_ARG, "bad arguments") : AFQ_ERR_ARG;
  afq::Mlp& m = c->mlp;
  if (!m.dims[0]) return fail(c, AFQ_ERR_STATE, "surrogate not initialised");
  if (m.n + n > m.cap) return fail(c, AFQ_ERR_ARG, "training set capacity exceeded");
  AFQ_GUARD_BEGIN
  const int F = m.dims[0];
  hip_check(scopy(c, m.X + m.n * F, X, (size_t)n * F * 4, hipMemcpyHostToDevice), "H2D");
  hip_check(scopy(c, m.Y + m.n, Y, (size_t)n * 4, hipMemcpyHostToDevice), "H2D");
  m.n += n;
  if (total) *total = m.n;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_surrogate_train(afq_ctx* c, int32_t epochs, int32_t batch, double lr, uint64_t seed, double* train_rmse,
                        double* valid_rmse) {
  if (!c || !c->mlp.dims[0]) return c ? fail(c, AFQ_ERR_STATE, "surrogate not initialised") : AFQ_ERR_ARG;
  afq::Mlp& m = c->mlp;
  if (m.n < 16) return fail(c, AFQ_ERR_STATE, "not enough training samples");
  if (batch <= 0 || batch > m.Bcap) return fail(c, AFQ_ERR_ARG, "bad batch size");
  AFQ_GUARD_BEGIN
  const int F = m.dims[0];
  const int64_t n = m.n;
  // standardisation from the data
  std::vector<float> X((size_t)n * F), Y(n);
  hip_check(scopy(c, X.data(), m.X, X.size() * 4, hipMemcpyDeviceToHost), "D2H");
  hip_check(scopy(c, Y.data(), m.Y, Y.size() * 4, hipMemcpyDeviceToHost), "D2H");
  // validation = the most recent tenth of the samples (collection order): the
  // same walker appears in consecutive steps with nearly the same features and
  // target, so a random split would hold out near-copies of training samples
  std::vector<int> perm(n);
  std::iota(perm.begin(), perm.end(), 0);
  std::mt19937_64 rng(seed);
  const int64_t nval = std::max<int64_t>(1, n / 10), ntr = n - nval;
  std::shuffle(perm.begin(), perm.begin() + ntr, rng);
  std::vector<double> mu(F, 0.0), var(F, 0.0);
  double ym = 0.0, yv = 0.0;
  for (int64_t q = 0; q < ntr; ++q) {
    const float* x = &X[(size_t)perm[q] * F];
    for (int f = 0; f < F; ++f) mu[f] += x[f];
    ym += Y[perm[q]];
  }
  for (int f = 0; f < F; ++f) mu[f] /= ntr;
  ym /= ntr;
  for (int64_t q = 0; q < ntr; ++q) {
    const float* x = &X[(size_t)perm[q] * F];
    for (int f = 0; f < F; ++f) var[f] += (x[f] - mu[f]) * (x[f] - mu[f]);
    yv += (Y[perm[q]] - ym) * (Y[perm[q]] - ym);
  }
  std::vector<float> muf(F), sdf(F);
  for (int f = 0; f < F; ++f) {
    muf[f] = (float)mu[f];
    const double sdv = std::sqrt(var[f] / ntr);
    sdf[f] = (float)(sdv > 1e-8 ? sdv : 1.0);
  }
  hip_check(scopy(c, m.mu, muf.data(), F * 4, hipMemcpyHostToDevice), "H2D");
  hip_check(scopy(c, m.sd, sdf.data(), F * 4, hipMemcpyHostToDevice), "H2D");
  m.t_mu = (float)ym;
  m.t_sd = (float)std::max(std::sqrt(yv / ntr), 1e-8);
  // didx[0, ntr): training indices (reshuffled every epoch); didx[ntr, n): validation
  int* didx = dalloc<int>(n);
  std::vector<float*> best;
  auto release = [&]() {
    (void)hipFree(didx);
    for (float* p : best) (void)hipFree(p);
  };
  try {
    hip_check(scopy(c, didx, perm.data(), n * sizeof(int), hipMemcpyHostToDevice), "H2D");
    // predictions (Ha) and targets of cnt samples listed at idx (device)
    auto predict = [&](const int* idx, int64_t cnt, std::vector<double>& pred, std::vector<double>& targ) {
      std::vector<float> y(std::min<int64_t>(cnt, m.Bcap));
      std::vector<int> ih(cnt);
      pred.resize(cnt);
      targ.resize(cnt);
      hip_check(scopy(c, ih.data(), idx, cnt * sizeof(int), hipMemcpyDeviceToHost), "D2H");
      for (int64_t b0 = 0; b0 < cnt; b0 += m.Bcap) {
        const int B = (int)std::min<int64_t>(m.Bcap, cnt - b0);
        afq::mlp_forward(m, m.X, idx + b0, B, c->stream);
        hip_check(hipMemcpyAsync(y.data(), m.h[3], B * 4, hipMemcpyDeviceToHost, c->stream), "D2H");
        hip_check(hipStreamSynchronize(c->stream), "sync");
        for (int q = 0; q < B; ++q) {
          pred[b0 + q] = (double)y[q] * m.t_sd + m.t_mu;
          targ[b0 + q] = Y[ih[b0 + q]];
        }
      }
    };
    auto rmse = [&](const int* idx, int64_t cnt) {
      std::vector<double> p, t;
      predict(idx, cnt, p, t);
      double acc = 0.0;
      for (int64_t q = 0; q < cnt; ++q) acc += (p[q] - t[q]) * (p[q] - t[q]);
      return std::sqrt(acc / cnt);
    };
    // the weights of the epoch with the lowest validation error are kept
    auto snapshot = [&](bool restore) {
      for (int l = 0, k = 0; l < 4; ++l)
        for (int wb = 0; wb < 2; ++wb, ++k) {
          const size_t bytes = 4 * (size_t)(wb == 0 ? m.dims[l] * m.dims[l + 1] : m.dims[l + 1]);
          float* live = wb == 0 ? m.w[l] : m.b[l];
          if ((int)best.size() <= k) best.push_back(dalloc<float>(bytes / 4));
          hip_check(hipMemcpyAsync(restore ? live : best[k], restore ? best[k] : live, bytes,
                                   hipMemcpyDeviceToDevice, c->stream), "D2D");
        }
    };
    double best_va = rmse(didx + ntr, nval);
    snapshot(false);
    std::vector<int> tr(perm.begin(), perm.begin() + ntr);
    for (int ep = 0; ep < epochs; ++ep) {
      std::shuffle(tr.begin(), tr.end(), rng);
      hip_check(hipMemcpyAsync(didx, tr.data(), ntr * sizeof(int), hipMemcpyHostToDevice, c->stream), "H2D");
      for (int64_t b0 = 0; b0 + batch <= ntr; b0 += batch) {
        afq::mlp_forward(m, m.X, didx + b0, batch, c->stream);
        afq::mlp_loss(m, m.Y, didx + b0, batch, c->stream);
        afq::mlp_backward(m, batch, c->stream);
        afq::mlp_adam(m, (float)lr, c->stream);
      }
      launch_check("train");
      const double va = rmse(didx + ntr, nval);
      if (va < best_va) {
        best_va = va;
        snapshot(false);
      }
    }
    snapshot(true);
    // Calibration on the validation set: the output becomes a + b * (network),
    // b = max(0, cov(y, p) / var(p)), the least-squares control-variate
    // coefficient; a network that predicts nothing falls back to the constant a.
    {
      std::vector<double> p, t;
      predict(didx + ntr, nval, p, t);
      double pm = 0.0, tm = 0.0, cpt = 0.0, vp = 0.0;
      for (int64_t q = 0; q < nval; ++q) { pm += p[q]; tm += t[q]; }
      pm /= nval;
      tm /= nval;
      for (int64_t q = 0; q < nval; ++q) {
        cpt += (p[q] - pm) * (t[q] - tm);
        vp += (p[q] - pm) * (p[q] - pm);
      }
      const double bcal = vp > 0.0 ? std::max(0.0, cpt / vp) : 0.0;
      const double acal = tm - bcal * pm;
      m.t_mu = (float)(acal + bcal * m.t_mu);
      m.t_sd = (float)(bcal * m.t_sd);
      m.calib_b = bcal;
    }
    if (train_rmse) *train_rmse = rmse(didx, ntr);
    if (valid_rmse) *valid_rmse = rmse(didx + ntr, nval);
    hip_check(hipStreamSynchronize(c->stream), "sync");
  } catch (...) {
    release();
    throw;
  }
  release();
  m.ready = true;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_surrogate_predict(afq_ctx* c, double* pred) {
  if (!c || !c->mlp.dims[0]) return c ? fail(c, AFQ_ERR_STATE, "surrogate not initialised") : AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  ensure_theta(c);
  afq::launch_features(s, nullptr, s.W, c->cvX, 0, c->stream);
  afq::launch_predict(s, c->mlp, c->cvX, s.W, c->cvS, c->stream);
  launch_check("predict");
  if (pred) download(pred, c->cvS, s.W, c->stream);
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_surrogate_params(afq_ctx* c, float* buf, int64_t nbuf, int32_t set) {
  if (!c || !c->mlp.dims[0]) return c ? fail(c, AFQ_ERR_STATE, "surrogate not initialised") : AFQ_ERR_ARG;
  afq::Mlp& m = c->mlp;
  const int F = m.dims[0];
  const int64_t need = mlp_nparams(m) + 2 * F + 2;
  if (!buf) return (int)AFQ_ERR_ARG;
  if (nbuf < need) return fail(c, AFQ_ERR_ARG, "buffer too small: need " + std::to_string(need));
  AFQ_GUARD_BEGIN
  int64_t off = 0;
  auto xfer = [&](float* d, int64_t cnt) {
    if (set) hip_check(scopy(c, d, buf + off, cnt * 4, hipMemcpyHostToDevice), "H2D");
    else hip_check(scopy(c, buf + off, d, cnt * 4, hipMemcpyDeviceToHost), "D2H");
    off += cnt;
  };
  for (int l = 0; l < 4; ++l) {
    xfer(m.w[l], (int64_t)m.dims[l] * m.dims[l + 1]);
    xfer(m.b[l], m.dims[l + 1]);
  }
  xfer(m.mu, F);
  xfer(m.sd, F);
  if (set) { m.t_mu = buf[off]; m.t_sd = buf[off + 1]; m.ready = true; }
  else { buf[off] = m.t_mu; buf[off + 1] = m.t_sd; }
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_surrogate_grad(afq_ctx* c, const float* X, const float* t, int32_t B, float* grads, double* loss) {
  if (!c || !c->mlp.dims[0]) return c ? fail(c, AFQ_ERR_STATE, "surrogate not initialised") : AFQ_ERR_ARG;
  afq::Mlp& m = c->mlp;
  if (!X || !t || B <= 0 || B > m.Bcap) return fail(c, AFQ_ERR_ARG, "bad batch");
  AFQ_GUARD_BEGIN
  const int F = m.dims[0];
  float* dX = dalloc<float>((int64_t)B * F);
  float* dT = dalloc<float>(B);
  hip_check(scopy(c, dX, X, (size_t)B * F * 4, hipMemcpyHostToDevice), "H2D");
  hip_check(scopy(c, dT, t, (size_t)B * 4, hipMemcpyHostToDevice), "H2D");
  afq::mlp_forward(m, dX, nullptr, B, c->stream);
  const float l = afq::mlp_loss(m, dT, nullptr, B, c->stream);
  afq::mlp_backward(m, B, c->stream);
  launch_check("grad");
  int64_t off = 0;
  for (int l2 = 0; l2 < 4; ++l2) {
    const int64_t nw = (int64_t)m.dims[l2] * m.dims[l2 + 1];
    hip_check(scopy(c, grads + off, m.gw[l2], nw * 4, hipMemcpyDeviceToHost), "D2H");
    off += nw;
    hip_check(scopy(c, grads + off, m.gb[l2], m.dims[l2 + 1] * 4, hipMemcpyDeviceToHost), "D2H");
    off += m.dims[l2 + 1];
  }
  if (loss) *loss = l;
  (void)hipFree(dX);
  (void)hipFree(dT);
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_energy_parts(afq_ctx* c, double* e1, double* ek) {
  if (!c || !c->last_exact_all) return c ? fail(c, AFQ_ERR_STATE, "needs an exact measurement of every walker") : AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  if (e1) {
    std::vector<double> v(2 * (size_t)s.W * s.nslots);
    download(v.data(), s.e1, v.size(), c->stream);
    for (int w = 0; w < s.W; ++w) {
      double a = 0.0;
      for (int q = 0; q < s.nslots; ++q) a += s.slot[q].mult * v[2 * ((size_t)w * s.nslots + q)];
      e1[w] = a;
    }
  }
  if (ek) {
    double* d = dalloc<double>(s.W);
    afq::launch_ek(s, nullptr, s.W, d, nullptr, 0, c->stream);
    launch_check("ek");
    download(ek, d, s.W, c->stream);
    (void)hipFree(d);
    // the exact measurement skips the exchange of walkers of weight zero: no E_K for them
    std::vector<double> w(s.W);
    download(w.data(), s.weights, s.W, c->stream);
    for (int i = 0; i < s.W; ++i)
      if (w[i] == 0.0) ek[i] = 0.0;
  }
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_surrogate_features(afq_ctx* c, float* X) {
  if (!c || !X) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  const int F = s.G + 2 * s.N;
  ensure_theta(c);
  float* d = dalloc<float>((int64_t)s.W * F);
  afq::launch_features(s, nullptr, s.W, d, 0, c->stream);
  launch_check("features");
  hip_check(scopy(c, X, d, (size_t)s.W * F * 4, hipMemcpyDeviceToHost), "D2H");
  (void)hipFree(d);
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_set_cv(afq_ctx* c, int32_t subset_inv, double risk_frac, double fallback_rms, uint64_t seed) {
  if (!c || subset_inv < 1) return c ? fail(c, AFQ_ERR_ARG, "subset_inv must be >= 1") : AFQ_ERR_ARG;
  if (!(risk_frac >= 0.0 && risk_frac <= 1.0)) return fail(c, AFQ_ERR_ARG, "risk_frac must lie in [0, 1]");
  AFQ_GUARD_BEGIN
  c->cv_minv = subset_inv;
  c->cv_risk = risk_frac;
  c->cv_fallback = fallback_rms;
  c->cv_seed = seed;
  c->cv_draw = 0;
  afq::launch_fill(c->s.stats + afq::SS_CVOFF, 1, 0.0, c->stream);   // the running offset starts at zero
  launch_check("cv offset");
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_debug_cv_force_position(afq_ctx* c, int32_t position) {
  if (!c) return AFQ_ERR_ARG;
  c->cv_force = position < 0 ? -1 : position;
  return AFQ_OK;
}

int afq_set_surrogate_kind(afq_ctx* c, int32_t kind, int32_t prec) {
  if (!c) return AFQ_ERR_ARG;
  if (kind != AFQ_SURR_MLP && kind != AFQ_SURR_EXCHANGE) return fail(c, AFQ_ERR_ARG, "unknown surrogate kind");
  if (kind == AFQ_SURR_EXCHANGE && prec != AFQ_PREC_BF16 && prec != AFQ_PREC_BF16X3 && prec != AFQ_PREC_FP8)
    return fail(c, AFQ_ERR_UNSUPPORTED, "surrogate exchange precision must be BF16, BF16X3 or FP8");
  AFQ_GUARD_BEGIN
  if (kind == AFQ_SURR_EXCHANGE) ensure_exchange_prec(c->s, prec, c->stream);
  ensure_cv(c);
  c->cv_kind = kind;
  c->cv_prec = prec;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_set_energy_clip(afq_ctx* c, const double* center, double halfwidth) {
  if (!c) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  ensure_cv(c);
  if (!center || !(halfwidth > 0.0)) {
    c->cv_halfw = 0.0;
    return AFQ_OK;
  }
  if (!c->cvCenter) c->cvCenter = dalloc<double>(c->s.W);
  hip_check(scopy(c, c->cvCenter, center, c->s.W * sizeof(double), hipMemcpyHostToDevice), "H2D");
  c->cv_nwr = 1;
  c->cv_halfw = halfwidth;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_set_clip_centers(afq_ctx* c, const double* centers, int32_t ncenters, double halfwidth) {
  if (!c) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  if (!centers || !(halfwidth > 0.0)) {
    c->cv_halfw = 0.0;
    return AFQ_OK;
  }
  if (ncenters < 1 || c->s.W % ncenters != 0)
    return fail(c, AFQ_ERR_ARG, "ncenters must divide the number of walkers");
  if (!c->cvCenter) c->cvCenter = dalloc<double>(c->s.W);
  // a small copy in stream order (no wait for the work already queued)
  hip_check(hipMemcpyAsync(c->cvCenter, centers, ncenters * sizeof(double), hipMemcpyHostToDevice, c->stream), "H2D");
  c->cv_nwr = c->s.W / ncenters;
  c->cv_halfw = halfwidth;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_block_totals(afq_ctx* c) {
  if (!c) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  const bool clip = !c->last_measure_clipped && c->cv_halfw > 0.0 && c->cvCenter;
  afq::launch_block_totals(c->s, c->cvCenter, c->cv_nwr, c->cv_halfw, clip, c->s.stats, c->stream);
  launch_check("block totals");
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_get_step_stats(afq_ctx* c, afq_step_stats* out) {
  if (!c || !out) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  double v[afq::STATS_DOUBLES];
  readback(c, {{v, c->s.stats, afq::STATS_DOUBLES}});
  out->total_weight = v[afq::SS_SUMW];
  out->n_propagated = (int64_t)v[afq::SS_NPROP];
  out->n_live = (int64_t)v[afq::SS_NLIVE];
  out->n_capped = (int64_t)v[afq::SS_NCAP];
  out->block_weight = v[afq::SS_BW];
  out->block_wsum = v[afq::SS_BWE];
  out->block_var = v[afq::SS_BVAR];
  out->n_measured = (int64_t)v[afq::SS_NMEAS];
  out->n_clipped = (int64_t)v[afq::SS_NCLIP];
  out->n_nonfinite = (int64_t)v[afq::SS_NBAD];
  out->n_exact = (int64_t)v[afq::SS_NEXACT];
  out->cv_rms = v[afq::SS_CVRMS];
  out->cv_var_sub = c->cv_last_fallback ? 0.0 : v[afq::SS_CVVAR];
  out->cv_mean_resid = v[afq::SS_CVMEAN];
  out->cv_fallback = c->cv_last_fallback ? 1 : 0;
  out->comb_total = v[afq::SS_COMB];
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_cv_stats(afq_ctx* c, double* out6) {
  if (!c || !out6) return AFQ_ERR_ARG;
  afq_step_stats t{};
  const int rc = afq_get_step_stats(c, &t);
  if (rc) return rc;
  out6[0] = (double)t.n_exact;
  out6[1] = t.cv_rms;
  out6[2] = t.cv_fallback;
  out6[3] = t.cv_var_sub;
  out6[4] = t.cv_mean_resid;
  out6[5] = (double)c->cv_nfallback;
  return AFQ_OK;
}

int afq_set_walkers_uniform(afq_ctx* c, const double* det, const double* overlap, double weight) {
  if (!c || !det) return c ? fail(c, AFQ_ERR_ARG, "null det") : AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  // one walker's block into the comb buffer, then into every walker
  upload(s.psi2, det, 2 * (size_t)s.ms, c->stream);
  afq::launch_broadcast_det(s, s.psi2, c->stream);
  afq::launch_fill(s.weights, s.W, weight, c->stream);
  if (overlap) {
    const std::complex<double> o(overlap[0], overlap[1]);
    std::vector<double> lo(2 * (size_t)s.W);
    for (int w = 0; w < s.W; ++w) {
      lo[2 * w] = std::log(std::abs(o));
      lo[2 * w + 1] = std::arg(o);
    }
    upload(s.logO, lo.data(), lo.size(), c->stream);
  }
  refresh_walkers(c, overlap == nullptr);
  launch_check("set_walkers_uniform");
  hip_check(hipStreamSynchronize(c->stream), "set_walkers_uniform sync");
  c->have_walkers = true;
  c->fb_stale = false;
  c->last_exact_all = false;
  c->last_measure_clipped = false;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_sync(afq_ctx* c) {
  if (!c) return AFQ_ERR_ARG;
  AFQ_GUARD_BEGIN
  hip_check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

}  // extern "C"

// ---------------------------------------------------------------- autotuner
// Times the variants of the whole propagation (both one-body factors and the series) on
// this context's current walkers and keeps the fastest: in FP64 k_vmul's 64 x 128 real tiles
// and k_taylor's 128 x 128-complex tiles, each between the one-body products, and, where it
// applies, the fused k_prop64; in split BF16 the two row tiles and the fused kernel.  The
// results go to the scratch t1, so the walkers stay as they are.
int afq_autotune(afq_ctx* c, int32_t* choice, double* ms_out) {
  if (!c) return AFQ_ERR_ARG;
  if (!c->prepped || !c->have_walkers) return fail(c, AFQ_ERR_STATE, "afq_prep_prop and afq_set_walkers first");
  AFQ_GUARD_BEGIN
  DevState& s = c->s;
  hipEvent_t a, b;
  hip_check(hipEventCreate(&a), "event");
  hip_check(hipEventCreate(&b), "event");
  double ms[4] = {0.0, 0.0, 0.0, 0.0};   // of variants 1 .. 3
  const int keep = s.taylor_variant;
  const bool split = s.prec_prop != AFQ_PREC_FP64;
  const int nv = (split ? afq::prop_fused_fits(s) : afq::prop64_fits(s)) ? 3 : 2;
  try {
    for (int v = 1; v <= nv; ++v) {
      s.taylor_variant = v;
      afq::launch_propagate_to(s, s.t1, c->stream);  // warm
      hip_check(hipEventRecord(a, c->stream), "record");
      for (int r = 0; r < 3; ++r) afq::launch_propagate_to(s, s.t1, c->stream);
      hip_check(hipEventRecord(b, c->stream), "record");
      hip_check(hipEventSynchronize(b), "sync");
      float t = 0.f;
      hip_check(hipEventElapsedTime(&t, a, b), "elapsed");
      ms[v] = t / 3.0;
    }
  } catch (...) {
    s.taylor_variant = keep;
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    throw;
  }
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  int pick = ms[2] < ms[1] ? 2 : 1;
  if (split && nv == 3 && ms[3] < ms[pick]) pick = 3;
  // FP64: choice and ms3 name the two tile shapes; the fused kernel is the shape rule's own (0)
  s.taylor_variant = !split && nv == 3 && ms[3] < ms[pick] ? 0 : pick;
  if (choice) *choice = pick;
  if (ms_out)
    for (int v = 1; v <= 3; ++v) ms_out[v - 1] = split || v < 3 ? ms[v] : 0.0;
  return AFQ_OK;
  AFQ_GUARD_END(c)
}

int afq_set_exchange_variant(afq_ctx* c, int32_t v) {
  if (!c || v < 0 || v > 4) return c ? fail(c, AFQ_ERR_ARG, "exchange variant must be 0 .. 4") : AFQ_ERR_ARG;
  c->s.xc_variant = v;
  return AFQ_OK;
}

int afq_set_vhs_tile(afq_ctx* c, int32_t v) {
  if (!c || v < 0 || v > 4) return c ? fail(c, AFQ_ERR_ARG, "VHS tile must be 0 .. 4") : AFQ_ERR_ARG;
  c->s.vhs_tile = v;
  return AFQ_OK;
}

int afq_set_exchange3_variant(afq_ctx* c, int32_t v) {
  if (!c || v < 0 || v > 2) return c ? fail(c, AFQ_ERR_ARG, "three-pass exchange variant must be 0, 1 or 2") : AFQ_ERR_ARG;
  c->s.xc3_variant = v;
  return AFQ_OK;
}

int afq_set_exchange64_variant(afq_ctx* c, int32_t v) {
  if (!c || v < 0 || v > 2) return c ? fail(c, AFQ_ERR_ARG, "FP64 exchange variant must be 0, 1 or 2") : AFQ_ERR_ARG;
  c->s.xc64_variant = v;
  return AFQ_OK;
}

int afq_set_exchange_chunks(afq_ctx* c, int32_t chunks) {
  if (!c || chunks < 0 || chunks > 4096) return c ? fail(c, AFQ_ERR_ARG, "chunks must lie in [0, 4096]") : AFQ_ERR_ARG;
  c->s.xc_chunks = chunks;
  return AFQ_OK;
}

int afq_set_force_bias_variant(afq_ctx* c, int32_t v) {
  if (!c || v < 0 || v > 1) return c ? fail(c, AFQ_ERR_ARG, "force bias variant must be 0 or 1") : AFQ_ERR_ARG;
  c->s.fb_split = v == 0;
  return AFQ_OK;
}

int afq_set_taylor_variant(afq_ctx* c, int32_t v) {
  if (!c || v < 0 || v > 3) return c ? fail(c, AFQ_ERR_ARG, "taylor variant must be 0, 1, 2 or 3") : AFQ_ERR_ARG;
  c->s.taylor_variant = v;
  return AFQ_OK;
}

// ---------------------------------------------------------------- batched systems
// Many independent populations (systems of different sizes) advanced together.
// One step of every system (propagation, optional QR, exact measurement of every
// walker, block totals with the clip, comb) is captured once into a hipGraph; a step
// is then one graph launch.  The step counter, energy shifts, comb uniforms and clip
// centres live in device arrays that the host refreshes between launches; block
// totals come back in one copy.
//
// Two forms of the captured step:
//  * grouped (default): every system's step is recorded launch by launch (the same
//    launchers as a single system's step, with a Recorder installed), stage by stage.
//    Within a stage the i-th launches of all systems that run the same kernel with the
//    same block shape become one launch of its grouped form over the concatenated
//    grids: one launch per stage and kernel for all systems (more only where systems'
//    shapes pick different kernels).  The systems can also be dealt over several lanes
//    (in decreasing size, so the lanes carry similar work), each grouped on its own
//    stream so that different stages of different lanes overlap; one lane is the
//    default (on the 64-system workload 4 lanes measured 3% slower than 1);
//  * branches (lanes = 0): each system's kernels on its own stream, forked from and
//    joined into the origin stream (one graph branch per system).
struct GroupLaunch {
  const void* fn = nullptr;
  dim3 block;
  unsigned shm = 0;
  uint32_t nblocks = 0;
  size_t ent_off = 0;   // index of its first GroupEntry in the batch's entry array
  size_t blk_off = 0;   // index of its first BlockRec in the batch's workgroup array
};
constexpr int kMaxLanes = 8;
struct afq_batch {
  std::vector<afq_ctx*> ctx;
  hipStream_t origin = nullptr;
  hipEvent_t fork = nullptr;
  std::vector<hipEvent_t> join;
  hipGraph_t graph[2] = {nullptr, nullptr};
  hipGraphExec_t exec[2] = {nullptr, nullptr};  // [0] plain step, [1] step with QR
  unsigned long long* d_step = nullptr;
  double* d_par = nullptr;   // [eshift | zeta | centre] x nsys
  double* d_tot = nullptr;   // 4 x nsys: sum w, sum w E, walkers propagated, walkers live
  double* h_par = nullptr;   // pinned staging of d_par
  double* h_tot = nullptr;   // pinned staging of d_tot
  double halfw = 0.0;
  uint64_t seed = 0;
  int ortho = 0;
  bool captured = false;
  bool stepped = false;   // h_tot holds the last step's totals
  int lanes = 1;   // grouped form on this many streams; 0: one graph branch per system
  // grouped form, per lane: [0] plain step, [1] step with QR
  std::vector<std::vector<GroupLaunch>> plan[2];
  std::vector<hipStream_t> lane_st;
  std::vector<hipEvent_t> lane_join;
  afq::GroupEntry* d_ent = nullptr;
  afq::BlockRec* d_blk = nullptr;
  unsigned char* d_packs = nullptr;
};

static void batch_enqueue(afq_batch* b, int i, bool qr) {
  afq_ctx* c = b->ctx[i];
  DevState& s = c->s;
  const int n = (int)b->ctx.size();
  hipStream_t st = c->stream;
  // afq::rec_stage() marks the stages the grouped form aligns across systems (the
  // same marks for every system, whatever its kernels)
  afq::rec_stage();
  afq::launch_fields(s, nullptr, b->seed + 7919ull * (uint64_t)i, 0, st);
  afq::rec_stage();
  if (s.prec_vhs == AFQ_PREC_FP64) afq::launch_vhs(s, st);
  else afq::launch_vhs_lp(s, s.prec_vhs, st);
  afq::rec_stage();
  afq::launch_expmul_pre(s, st);
  afq::launch_taylor(s, st);
  afq::launch_expmul_post(s, st);
  afq::rec_stage();
  afq::launch_green(s, false, st);
  afq::launch_weight(s, 0.0, true, st);
  afq::rec_stage();
  run_force_bias(s, st);
  afq::rec_stage();
  if (qr) afq::launch_qr(s, st);
  afq::rec_stage();
  if (s.GE > 0) {
    if (s.prec_exchange == AFQ_PREC_FP64) afq::launch_exchange(s, nullptr, s.W, st);
    else afq::launch_exchange_lp(s, nullptr, s.W, s.prec_exchange, st);
  }
  afq::rec_stage();
  afq::launch_energy(s, nullptr, s.W, 0.0, st);
  afq::launch_block_energy(s, b->d_par + 2 * n + i, b->halfw, b->d_tot + 4 * i, st);
  afq::rec_stage();
  afq::launch_comb(s, 0.0, st);
  launch_check("batch step");
}

// Points system i's per-step inputs at the batch's device arrays for recording or
// capture (and back afterwards).
static void batch_bind(afq_batch* b, int i, bool on) {
  DevState& s = b->ctx[i]->s;
  const int n = (int)b->ctx.size();
  s.d_step = on ? b->d_step : nullptr;
  s.d_eshift = on ? b->d_par + i : nullptr;
  s.d_zeta = on ? b->d_par + n + i : nullptr;
  s.graph_mode = on;
}

// The grouped form of one step: every system's launches recorded, then grouped by
// (stage, position in the stage, grouped kernel, block, LDS).  Entries and argument
// packs of both plans go to one device allocation each.
static void batch_plan(afq_batch* b, std::vector<afq::GroupEntry>& ents, std::vector<afq::BlockRec>& blks,
                       std::vector<unsigned char>& packs) {
  const int n = (int)b->ctx.size();
  for (int k = 0; k < 2; ++k) {
    std::vector<afq::Recorder> rec(n);
    for (int i = 0; i < n; ++i) {
      afq_ctx* c = b->ctx[i];
      // a launch that does not go through the recorder would land in this capture
      hip_check(hipStreamBeginCapture(c->stream, hipStreamCaptureModeRelaxed), "hipStreamBeginCapture");
      batch_bind(b, i, true);
      afq::g_recorder = &rec[i];
      hipGraph_t stray = nullptr;
      try {
        batch_enqueue(b, i, k == 1);
      } catch (...) {
        afq::g_recorder = nullptr;
        batch_bind(b, i, false);
        (void)hipStreamEndCapture(c->stream, &stray);
        if (stray) (void)hipGraphDestroy(stray);
        throw;
      }
      afq::g_recorder = nullptr;
      batch_bind(b, i, false);
      hip_check(hipStreamEndCapture(c->stream, &stray), "hipStreamEndCapture");
      size_t nodes = 0;
      const hipError_t e = hipGraphGetNodes(stray, nullptr, &nodes);
      (void)hipGraphDestroy(stray);
      hip_check(e, "hipGraphGetNodes");
      if (nodes != 0)
        throw DevError(AFQ_ERR_DEVICE, "a kernel of the batched step was launched outside the grouped path");
      rec[i].stage_starts.push_back(rec[i].recs.size());
      if (rec[i].stage_starts.size() != rec[0].stage_starts.size())
        throw DevError(AFQ_ERR_DEVICE, "systems recorded different numbers of stages");
    }
    std::vector<int> order(n);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
      const DevState& a = b->ctx[x]->s;
      const DevState& c = b->ctx[y]->s;
      return (int64_t)a.N * a.G > (int64_t)c.N * c.G;
    });
    // the systems dealt over the lanes in decreasing size, so the lanes carry similar work
    const int L = std::min(b->lanes, n);
    b->plan[k].assign(L, {});
    for (int lane = 0; lane < L; ++lane) {
    std::vector<GroupLaunch>& plan = b->plan[k][lane];
    std::vector<int> mine;
    for (int j = lane; j < n; j += L) mine.push_back(order[j]);
    const size_t nst = rec[0].stage_starts.size() - 1;
    for (size_t t = 0; t < nst; ++t) {
      size_t depth = 0;
      for (int i : mine) depth = std::max(depth, rec[i].stage_starts[t + 1] - rec[i].stage_starts[t]);
      for (size_t l = 0; l < depth; ++l) {
        // the l-th launch of this stage of every system that has one, grouped by kernel;
        // the systems in decreasing size, so that the workgroups that run longest are
        // dispatched first and do not form the launch's tail
        std::vector<std::vector<const afq::LaunchRec*>> groups;
        for (int i : mine) {
          const size_t j = rec[i].stage_starts[t] + l;
          if (j >= rec[i].stage_starts[t + 1]) continue;
          const afq::LaunchRec* r = &rec[i].recs[j];
          bool placed = false;
          for (auto& g : groups) {
            const afq::LaunchRec* q = g[0];
            if (q->fn == r->fn && q->shm == r->shm && q->block.x == r->block.x && q->block.y == r->block.y &&
                q->block.z == r->block.z) {
              g.push_back(r);
              placed = true;
              break;
            }
          }
          if (!placed) groups.push_back({r});
        }
        for (auto& g : groups) {
          GroupLaunch gl;
          gl.fn = g[0]->fn;
          gl.block = g[0]->block;
          gl.shm = g[0]->shm;
          gl.ent_off = ents.size();
          gl.blk_off = blks.size();
          uint64_t start = 0;
          for (const afq::LaunchRec* r : g) {
            const uint64_t nb = (uint64_t)r->grid.x * r->grid.y * r->grid.z;
            if (nb == 0) continue;
            if (start + nb >= (1ull << 31)) throw DevError(AFQ_ERR_UNSUPPORTED, "grouped launch too large");
            size_t off = (packs.size() + 15) & ~(size_t)15;
            if (r->align > 16) off = (off + r->align - 1) / r->align * r->align;
            packs.resize(off + r->pack.size());
            std::memcpy(packs.data() + off, r->pack.data(), r->pack.size());
            const uint32_t ei = (uint32_t)(ents.size() - gl.ent_off);
            afq::GroupEntry e;
            e.gx = r->grid.x;
            e.gy = r->grid.y;
            e.gz = r->grid.z;
            e.pad = 0;
            ents.push_back(e);
            for (uint64_t q = 0; q < nb; ++q) {
              afq::BlockRec br;
              br.ent = ei;
              br.local = (uint32_t)q;
              br.off = off;
              blks.push_back(br);
            }
            start += nb;
          }
          gl.nblocks = (uint32_t)start;
          if (gl.nblocks > 0) plan.push_back(gl);
        }
      }
    }
    }
  }
}

// the grouped step (captured or issued directly): each lane's launches on its own
// stream, forked from and joined back into the origin stream
static void batch_issue_grouped(afq_batch* b, bool qr) {
  const auto& lanes = b->plan[qr ? 1 : 0];
  hip_check(hipEventRecord(b->fork, b->origin), "record");
  for (size_t lane = 0; lane < lanes.size(); ++lane) {
    hipStream_t st = b->lane_st[lane];
    hip_check(hipStreamWaitEvent(st, b->fork, 0), "wait");
    for (const GroupLaunch& gl : lanes[lane]) {
      const afq::GroupEntry* ent = b->d_ent + gl.ent_off;
      const afq::BlockRec* blk = b->d_blk + gl.blk_off;
      const unsigned char* packs = b->d_packs;
      void* args[] = {(void*)&ent, (void*)&blk, (void*)&packs};
      hip_check(hipLaunchKernel(gl.fn, dim3(gl.nblocks), gl.block, args, gl.shm, st), "grouped launch");
    }
    hip_check(hipEventRecord(b->lane_join[lane], st), "record");
    hip_check(hipStreamWaitEvent(b->origin, b->lane_join[lane], 0), "wait");
  }
  afq::launch_step_inc(b->d_step, b->origin);
}

// all systems' step on their streams, forked from and joined back into the origin stream
static void batch_record(afq_batch* b, bool qr) {
  if (b->lanes > 0) {
    batch_issue_grouped(b, qr);
    return;
  }
  const int n = (int)b->ctx.size();
  hip_check(hipEventRecord(b->fork, b->origin), "record");
  for (int i = 0; i < n; ++i) {
    afq_ctx* c = b->ctx[i];
    batch_bind(b, i, true);
    hip_check(hipStreamWaitEvent(c->stream, b->fork, 0), "wait");
    try {
      batch_enqueue(b, i, qr);
    } catch (...) {
      batch_bind(b, i, false);
      throw;
    }
    batch_bind(b, i, false);
    hip_check(hipEventRecord(b->join[i], c->stream), "record");
    hip_check(hipStreamWaitEvent(b->origin, b->join[i], 0), "wait");
  }
  afq::launch_step_inc(b->d_step, b->origin);
}

static void batch_free(afq_batch* b) {
  for (int k = 0; k < 2; ++k) {
    if (b->exec[k]) (void)hipGraphExecDestroy(b->exec[k]);
    if (b->graph[k]) (void)hipGraphDestroy(b->graph[k]);
  }
  for (afq_ctx* c : b->ctx) afq_destroy(c);
  for (hipEvent_t e : b->join) (void)hipEventDestroy(e);
  for (hipEvent_t e : b->lane_join) (void)hipEventDestroy(e);
  for (hipStream_t st : b->lane_st) (void)hipStreamDestroy(st);
  if (b->fork) (void)hipEventDestroy(b->fork);
  if (b->origin) (void)hipStreamDestroy(b->origin);
  if (b->d_step) (void)hipFree(b->d_step);
  if (b->d_par) (void)hipFree(b->d_par);
  if (b->d_tot) (void)hipFree(b->d_tot);
  if (b->h_par) (void)hipHostFree(b->h_par);
  if (b->h_tot) (void)hipHostFree(b->h_tot);
  if (b->d_ent) (void)hipFree(b->d_ent);
  if (b->d_blk) (void)hipFree(b->d_blk);
  if (b->d_packs) (void)hipFree(b->d_packs);
  delete b;
}

int afq_batch_create(int32_t nsys, const afq_ham* hams, const afq_trial* trials, const afq_params* params,
                     afq_batch** out) {
  if (nsys <= 0 || !hams || !trials || !params || !out) return fail(nullptr, AFQ_ERR_ARG, "bad batch arguments");
  for (int i = 0; i < nsys; ++i)
    if (hams[i].h1_dn || hams[i].h1_mod_dn || hams[i].chol_dn)
      return fail(nullptr, AFQ_ERR_UNSUPPORTED, "batched systems take restricted integrals only");
  afq_batch* b = new afq_batch();
  for (int i = 0; i < nsys; ++i) {
    afq_ctx* c = nullptr;
    const int rc = afq_create(&hams[i], &trials[i], &params[i], &c);
    if (rc) {
      batch_free(b);
      return rc;
    }
    b->ctx.push_back(c);
  }
  try {
    hip_check(hipStreamCreateWithFlags(&b->origin, hipStreamNonBlocking), "stream");
    hip_check(hipEventCreateWithFlags(&b->fork, hipEventDisableTiming), "event");
    b->join.resize(nsys, nullptr);
    for (int i = 0; i < nsys; ++i) hip_check(hipEventCreateWithFlags(&b->join[i], hipEventDisableTiming), "event");
    b->lane_st.resize(kMaxLanes, nullptr);
    b->lane_join.resize(kMaxLanes, nullptr);
    for (int l = 0; l < kMaxLanes; ++l) {
      hip_check(hipStreamCreateWithFlags(&b->lane_st[l], hipStreamNonBlocking), "stream");
      hip_check(hipEventCreateWithFlags(&b->lane_join[l], hipEventDisableTiming), "event");
    }
    b->d_step = dalloc<unsigned long long>(1);
    b->d_par = dalloc<double>(3 * (size_t)nsys);
    b->d_tot = dalloc<double>(4 * (size_t)nsys);
    hip_check(hipHostMalloc((void**)&b->h_par, 3 * sizeof(double) * nsys, 0), "hipHostMalloc");
    hip_check(hipHostMalloc((void**)&b->h_tot, 4 * sizeof(double) * nsys, 0), "hipHostMalloc");
  } catch (const std::exception& e) {
    batch_free(b);
    return fail(nullptr, AFQ_ERR_DEVICE, e.what());
  }
  *out = b;
  return AFQ_OK;
}

int afq_batch_destroy(afq_batch* b) {
  if (!b) return AFQ_OK;
  if (b->origin) (void)hipStreamSynchronize(b->origin);
  batch_free(b);
  return AFQ_OK;
}

int afq_batch_context(afq_batch* b, int32_t i, afq_ctx** c) {
  if (!b || !c || i < 0 || i >= (int)b->ctx.size()) return fail(nullptr, AFQ_ERR_ARG, "bad system index");
  *c = b->ctx[i];
  return AFQ_OK;
}

int afq_batch_set_lanes(afq_batch* b, int32_t lanes) {
  if (!b || lanes < 0 || lanes > kMaxLanes) return fail(nullptr, AFQ_ERR_ARG, "lanes must be 0 .. 8");
  b->lanes = lanes;
  b->captured = false;   // the captured form changes: capture again
  return AFQ_OK;
}

int afq_batch_launches(afq_batch* b, int32_t qr, int32_t* launches) {
  if (!b || !launches) return fail(nullptr, AFQ_ERR_ARG, "bad launches arguments");
  if (!b->captured) return fail(nullptr, AFQ_ERR_STATE, "afq_batch_capture first");
  if (b->lanes == 0) {
    *launches = -1;
    return AFQ_OK;
  }
  int32_t nl = 1;   // the step counter
  for (const auto& lane : b->plan[qr ? 1 : 0]) nl += (int32_t)lane.size();
  *launches = nl;
  return AFQ_OK;
}

int afq_batch_capture(afq_batch* b, uint64_t seed, int32_t ortho_steps, double clip_halfwidth, uint64_t first_step) {
  if (!b || ortho_steps <= 0) return fail(nullptr, AFQ_ERR_ARG, "bad capture arguments");
  for (afq_ctx* c : b->ctx)
    if (!c->prepped || !c->have_walkers)
      return fail(nullptr, AFQ_ERR_STATE, "every system needs afq_prep_prop and afq_set_walkers first");
  try {
    for (afq_ctx* c : b->ctx) hip_check(hipStreamSynchronize(c->stream), "sync");
    b->seed = seed;
    b->ortho = ortho_steps;
    b->halfw = clip_halfwidth;
    if (b->d_ent) { (void)hipFree(b->d_ent); b->d_ent = nullptr; }
    if (b->d_blk) { (void)hipFree(b->d_blk); b->d_blk = nullptr; }
    if (b->d_packs) { (void)hipFree(b->d_packs); b->d_packs = nullptr; }
    b->plan[0].clear();
    b->plan[1].clear();
    if (b->lanes > 0) {
      std::vector<afq::GroupEntry> ents;
      std::vector<afq::BlockRec> blks;
      std::vector<unsigned char> packs;
      batch_plan(b, ents, blks, packs);
      b->d_ent = dalloc<afq::GroupEntry>(std::max<size_t>(1, ents.size()));
      b->d_blk = dalloc<afq::BlockRec>(std::max<size_t>(1, blks.size()));
      if (!blks.empty())
        hip_check(hipMemcpy(b->d_blk, blks.data(), blks.size() * sizeof(afq::BlockRec), hipMemcpyHostToDevice), "H2D");
      b->d_packs = dalloc<unsigned char>(std::max<size_t>(16, packs.size()));
      if (!ents.empty())
        hip_check(hipMemcpy(b->d_ent, ents.data(), ents.size() * sizeof(afq::GroupEntry), hipMemcpyHostToDevice), "H2D");
      if (!packs.empty())
        hip_check(hipMemcpy(b->d_packs, packs.data(), packs.size(), hipMemcpyHostToDevice), "H2D");
    }
    for (int k = 0; k < 2; ++k) {
      if (b->exec[k]) { (void)hipGraphExecDestroy(b->exec[k]); b->exec[k] = nullptr; }
      if (b->graph[k]) { (void)hipGraphDestroy(b->graph[k]); b->graph[k] = nullptr; }
      hip_check(hipStreamBeginCapture(b->origin, hipStreamCaptureModeGlobal), "hipStreamBeginCapture");
      try {
        batch_record(b, k == 1);
      } catch (...) {
        hipGraph_t g = nullptr;
        (void)hipStreamEndCapture(b->origin, &g);
        if (g) (void)hipGraphDestroy(g);
        throw;
      }
      hip_check(hipStreamEndCapture(b->origin, &b->graph[k]), "hipStreamEndCapture");
      hip_check(hipGraphInstantiate(&b->exec[k], b->graph[k], nullptr, nullptr, 0), "hipGraphInstantiate");
    }
    const unsigned long long s0 = first_step;
    hip_check(hipMemcpyAsync(b->d_step, &s0, sizeof(s0), hipMemcpyHostToDevice, b->origin), "H2D");
    hip_check(hipStreamSynchronize(b->origin), "sync");
    b->captured = true;
  } catch (const DevError& e) {
    return fail(nullptr, e.code, e.what());
  } catch (const std::exception& e) {
    return fail(nullptr, AFQ_ERR_DEVICE, e.what());
  }
  return AFQ_OK;
}

// One step of every system.  eshift / zeta / center: per system; totals receives
// {sum w, sum w clip(E_L)} per system (before the comb).  graph = 0 issues the same
// kernels one launch at a time (no capture) for comparison.
int afq_batch_step(afq_batch* b, int64_t step, const double* eshift, const double* zeta, const double* center,
                   int32_t graph, double* totals) {
  if (!b || !eshift || !zeta || !center || !totals) return fail(nullptr, AFQ_ERR_ARG, "bad step arguments");
  if (!b->captured) return fail(nullptr, AFQ_ERR_STATE, "afq_batch_capture first");
  const int n = (int)b->ctx.size();
  try {
    for (int i = 0; i < n; ++i) {
      b->h_par[i] = eshift[i];
      b->h_par[n + i] = zeta[i];
      b->h_par[2 * n + i] = center[i];
    }
    hip_check(hipMemcpyAsync(b->d_par, b->h_par, 3 * sizeof(double) * n, hipMemcpyHostToDevice, b->origin), "H2D");
    const bool qr = step % b->ortho == 0;
    if (graph) {
      hip_check(hipGraphLaunch(b->exec[qr ? 1 : 0], b->origin), "hipGraphLaunch");
    } else {
      batch_record(b, qr);
    }
    hip_check(hipMemcpyAsync(b->h_tot, b->d_tot, 4 * sizeof(double) * n, hipMemcpyDeviceToHost, b->origin), "D2H");
    hip_check(hipStreamSynchronize(b->origin), "sync");
    for (int i = 0; i < n; ++i) {
      totals[2 * i] = b->h_tot[4 * i];
      totals[2 * i + 1] = b->h_tot[4 * i + 1];
    }
    b->stepped = true;
  } catch (const DevError& e) {
    return fail(nullptr, e.code, e.what());
  } catch (const std::exception& e) {
    return fail(nullptr, AFQ_ERR_DEVICE, e.what());
  }
  return AFQ_OK;
}

int afq_batch_counts(afq_batch* b, int64_t* propagated, int64_t* live) {
  if (!b || !propagated || !live) return fail(nullptr, AFQ_ERR_ARG, "bad counts arguments");
  if (!b->stepped) return fail(nullptr, AFQ_ERR_STATE, "no afq_batch_step yet");
  for (size_t i = 0; i < b->ctx.size(); ++i) {
    propagated[i] = (int64_t)b->h_tot[4 * i + 2];
    live[i] = (int64_t)b->h_tot[4 * i + 3];
  }
  return AFQ_OK;
}
