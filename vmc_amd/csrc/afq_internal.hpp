// Internal declarations shared by the kernels (afq_kernels.hip) and the host
// context / C ABI (afq_ctx.cpp).  Not part of the public interface.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <random>
#include <string>
#include <vector>

#include "../../include/vmc_afqmc.h"

namespace afq {

// One spin slot of the trial evaluation.  An RHF walker against an RHF trial
// collapses to a single slot of multiplicity 2 (DQMC/RHF.cpp:80-107,150-177);
// every other pairing uses two slots of multiplicity 1.
struct Slot {
  int n;         // electrons in the slot
  int det;       // walker determinant it reads (0 or 1)
  int phi;       // trial orbital set (0 up, 1 down)
  int mult;      // multiplicity
  int64_t koff;  // offset of this slot in a walker's theta / the rotated Cholesky rows (complex / real elems)
};

// Per-kernel device time buckets (afq_stage_times order).
enum Stage { ST_FB = 0, ST_FIELDS, ST_VHS, ST_PROP, ST_GREEN, ST_WEIGHT, ST_ORTHO, ST_ENERGY, ST_COMB, ST_TAYLOR,
             ST_EXLP, ST_COUNT };

// Slots of DevState::stats, the device copy of the population statistics
// (afq_step_stats): step totals, block totals, control-variate numbers, the comb total.
enum StatSlot {
  SS_SUMW = 0, SS_NPROP, SS_NLIVE, SS_NCAP,                  // the last propagation
  SS_BW, SS_BWE, SS_BVAR, SS_NMEAS, SS_NCLIP, SS_NBAD,        // the last block totals
  SS_NEXACT, SS_CVRMS, SS_CVVAR, SS_CVMEAN, SS_CVOFF, SS_NRISK, SS_NRAND,  // the last control variate
  SS_COMB,                                                    // the last comb
  SS_COUNT_
};
constexpr int STATS_DOUBLES = 32;

// order of an FP64 force bias sum over k: units of ku (a multiple of 16), chunks of s units
struct FbOrder { int ku, s; };

struct DevState {
  // sizes
  int N = 0, na = 0, nb = 0, G = 0, GE = 0, W = 0;
  int64_t T = 0;        // N(N+1)/2
  int64_t ms = 0;       // complex elements per walker determinant set, N(na+nb)
  int64_t Ktot = 0;     // complex elements of theta per walker, sum_s N n_s
  int nslots = 0;
  Slot slot[2];
  int ndets_prop = 0;   // determinants propagated per walker (1 for an RHF walker)
  int det_n[2] = {0, 0};
  int64_t det_off[2] = {0, 0};  // complex offset of det d in a walker's serial block
  bool walker_rhf = false, trial_rhf = false, ref_compat = false;
  double ecore = 0.0, dt = 0.0, weight_cap = 100.0;
  double prop_const_re = 0.0, prop_const_im = 0.0;

  // unrestricted integrals (intType "u"): per-spin one-body propagator, Cholesky
  // vectors and VHS; E, Lp and P are then the up-spin ones, E2, Lp2 and P2 the
  // down-spin ones (FP64 VHS and propagation only)
  bool uints = false;
  double* E2 = nullptr; double* Lp2 = nullptr; double* P2 = nullptr;

  // Hamiltonian / trial (device)
  double* E = nullptr;      // exp(-dt/2 h1'), N x N
  double* Lp = nullptr;     // packed lower-triangle L, G x T (FP64, or float-rounded in ref_compat)
  double* R = nullptr;      // rotated Cholesky, G x Ktot: [g][koff_s + k*n_s + i] = (Phi_s^T L_g)(i,k)
  double* phi[2] = {nullptr, nullptr};   // N x n_s row-major
  double* hphi[2] = {nullptr, nullptr};  // h1 Phi_s, N x n_s
  double* mf = nullptr;     // G complex mean-field shifts

  // walkers (device)
  double* psi = nullptr;    // W x ms complex (serial layout)
  double* theta = nullptr;  // W x Ktot complex
  double* fb = nullptr;     // W x G complex
  double* logO = nullptr;   // W complex: log of the trial overlap
  double* e1 = nullptr;     // W x nslots complex one-body partial
  double* logdet = nullptr; // W x nslots complex, from the last Green's-function evaluation
  double* weights = nullptr;
  double* factors = nullptr;
  // comb double buffers
  double* psi2 = nullptr; double* theta2 = nullptr; double* fb2 = nullptr;
  double* logO2 = nullptr; double* e12 = nullptr;
  // step scratch
  double* fields = nullptr;  // W x G complex
  double* sft = nullptr;     // W x 4: shift (complex), fbTerm (complex)
  double* P = nullptr;       // W x 2 x N x N (VHS: sum_g Re/Im(field) L_g, both triangles)
  double* t0 = nullptr; double* t1 = nullptr; double* accb = nullptr;  // W x ms complex
  double* draws = nullptr;   // W x G (replay)
  double* Sg = nullptr;      // W x nslots x 64 x 128: overlap matrices S = Phi^T psi, then S^-1
  // FP64 force bias: partial sums over chunks of K.  Not a buffer of its own: it borrows
  // one that nothing reads between the Green's function and the end of the force bias,
  // the larger of Sg (S^-1 is used up by theta) and theta2 (live inside a comb only);
  // a temporary population borrows Sg, whichever entry point made it.  fbo is the order of
  // the sum, which is the same for all of them
  double* fbw = nullptr; int64_t fbw_doubles = 0;
  FbOrder fbo{};
  double* Xp = nullptr;      // nslots x W x ngt complex exchange partials
  int ngt_cap = 0;
  double* eloc = nullptr;    // W
  double* ho = nullptr;      // W x 4 {E*O, O}
  double* cum = nullptr;     // W (comb)
  int* idx = nullptr;        // W (comb)
  int* live = nullptr;       // W: walkers of nonzero weight in ascending order, count in *nlive
  int* nlive = nullptr;
  int* gfresh = nullptr;     // W: 1 where the last launch_green_pre took the walker
  unsigned long long* ncap = nullptr;   // [0] walkers capped, [1] walkers propagated in the last step
  double* stats = nullptr;   // STATS_DOUBLES: population statistics (StatSlot)

  // mixed precision
  int prec_exchange = AFQ_PREC_FP64;
  int Np = 0;               // N padded to a multiple of 8 (bf16 rows)
  int ctot = 0;             // theta columns per walker, 2 sum_s n_s
  unsigned short* Rb_hi = nullptr; unsigned short* Rb_lo = nullptr;  // [slot][g][i][Np]
  unsigned short* Tb_hi = nullptr; unsigned short* Tb_lo = nullptr;  // [w][re/im][slot][j][Np]
  // FP32 partial force bias of each slot, [slot][2W rows][G], for the two-slot split of
  // k_force_bias_bf16 (allocated with Tb_hi when there are two slots)
  float* fbp = nullptr;
  int fbp_rows = 0;
  // the hi part of R in MFMA fragment order for the pair-wise exchange (allocated with
  // Rb_hi where every slot has at most 64 electrons and N fits its LDS):
  // Rf[slot][g][ks][b][lane][8] = R_g[16 b + lane % 16][32 ks + 8 (lane / 16) + 0..7],
  // zero outside the data; rf_off[slot] is the slot's offset in u16
  unsigned short* Rf = nullptr;
  unsigned short* Rf_lo = nullptr;   // the lo parts, same layout (the three-pass exact level)
  int64_t rf_off[2] = {0, 0};
  int prec_fb = AFQ_PREC_FP64, prec_vhs = AFQ_PREC_FP64;
  // Tb holds the split theta of every walker of nonzero weight (set by the split-BF16
  // force bias; cleared by whatever changes theta or the weights), so the exchange of
  // the same walkers need not split again
  mutable bool tb_live = false;
  // Tb holds the split theta of the walkers the last launch_theta_post took (the fresh
  // ones still alive), written by that kernel; the next force bias splits only the rest
  mutable bool tb_post = false;
  // theta is not carried through an eager comb (nothing reads it before the next
  // step's Green's function recomputes it); entry points that read it first call
  // ensure_theta, and the next propagation recomputes it for every walker
  bool theta_stale = false;
  int prec_prop = AFQ_PREC_FP64;   // Taylor products V t
  // split-BF16 Taylor operands (allocated when prec_prop is BF16X3); orbitals come in
  // chunks of 16 (Nq = N padded to 16, pads stay zero):
  //   Vh/Vl  [w][chunk][i][32]: hi/lo of [-P_im | P_re] over the chunk's 16 orbitals
  //   Ub[0], Ub[1] (Horner terms) and Ub[2] (E psi): [w][plane][chunk][q][16], planes
  //          re_hi, re_lo, im_hi, im_lo; q runs over the na + nb propagated columns
  //   Dh/Dl  D = E - I (the one-body factor less the identity), N rows of pitch
  //          onebody_pitch(N)
  int Nq = 0;
  unsigned short* Vh = nullptr; unsigned short* Vl = nullptr;
  unsigned short* Ub[3] = {nullptr, nullptr, nullptr};
  unsigned short* Dh = nullptr; unsigned short* Dl = nullptr;
  // replayed (hipGraph) steps: step counter, energy shift and comb uniform live in
  // device memory, and the comb copies back instead of swapping buffers
  const unsigned long long* d_step = nullptr;
  const double* d_eshift = nullptr;
  const double* d_zeta = nullptr;
  bool graph_mode = false;
  // Taylor kernels: 0 by shape; FP64: 1 k_vmul (64 x 128 tiles), 2 k_taylor (128 x 128
  // complex), both between separate one-body products, else the fused k_prop64 (N <= 384); split BF16: 1 128-row tiles, 2 160-row tiles (one-body factors and Taylor
  // steps as separate kernels), 3 the fused k_prop_split (the default where N <= 384)
  int taylor_variant = 0;
  // one-pass BF16 exchange: 0 by shape (k_exchange_pw2 with 8 waves where it applies,
  // else k_exchange_pw, else the tiled kernel), 1 the tiled k_exchange_bf16,
  // 2 k_exchange_pw, 3 k_exchange_pw2 with 4 waves, 4 k_exchange_pw2 with 8 waves
  int xc_variant = 0;
  // three-pass split-BF16 exchange (the control variate's exact level): 0 by shape (the
  // pair-wise k_exchange_pw2<., 4, true> where it applies), 1 the tiled k_exchange_bf16<2>
  int xc3_variant = 0;
  // pair-wise exchange: chunks of the Cholesky vectors per (walker, slot); each chunk is
  // one workgroup, and the workgroups of all walkers take the chunks in the same order, so
  // a chunk of R streams through each XCD's L2 once per wave of resident workgroups
  // (0: by shape)
  int xc_chunks = 0;
  // FP64 exchange kernel: 0 by shape (k_exchange64 from 4 electrons a slot up, else
  // k_exchange2 with 8 waves), 1 k_exchange (element loaders), 2 k_exchange2 with 4 waves
  int xc64_variant = 0;
  // split-BF16 force bias: one workgroup per slot and FP64 combine (true, default), or
  // both slots in one workgroup
  bool fb_split = true;
  // split-BF16 VHS tile (k_vhs_bf16): 0 128 rows single-buffered, 1 256 rows
  // double-buffered, 2 128 rows double-buffered, 3 (default) and 4 as 0 and 2 with the
  // output below the diagonal staged through LDS and written in 16-byte runs
  int vhs_tile = 3;
  int Gp = 0;               // G padded to a multiple of 8
  unsigned short* Lt_hi = nullptr; unsigned short* Lt_lo = nullptr;  // packed L transposed, [t][Gp]
  unsigned short* Fb_hi = nullptr; unsigned short* Fb_lo = nullptr;  // fields, [w][re/im][Gp]
  // e4m3 exchange operands (allocated on first use): Rq8[slot][g][i][Npq] with 1/s_g in
  // rinv8[g]; Tq8[w][re/im][slot][j][Npq] with 1/t in tinv8[w][slot]; Npq = N padded to 16
  int Npq = 0;
  unsigned char* Rq8 = nullptr; unsigned char* Tq8 = nullptr;
  float* rinv8 = nullptr; float* tinv8 = nullptr;
  int* vhs_blk = nullptr;   // (i0, j0) of the 16 x 8 blocks of V that touch the lower triangle
  int nvhs_blk = 0;
};

// Exchange-energy surrogate: GELU MLP dims[0] -> dims[1] -> dims[2] -> dims[3] -> 1,
// FP32 master weights w[l] (dims[l] x dims[l+1], row-major), Adam moments,
// activation buffers for up to Bcap rows, and the training set (X: n x F, Y: n).
struct Mlp {
  int dims[5] = {0, 0, 0, 0, 0};
  float* w[4] = {}; float* b[4] = {};
  float* mw[4] = {}; float* vw[4] = {}; float* mb[4] = {}; float* vb[4] = {};
  float* gw[4] = {}; float* gb[4] = {};
  float* z[4] = {}; float* h[4] = {}; float* dh[4] = {};
  float* mu = nullptr; float* sd = nullptr;
  float t_mu = 0.f, t_sd = 1.f;
  float* lossbuf = nullptr;
  float* xn = nullptr;   // standardised input rows of the batch, Bcap x F
  float* ws = nullptr;   // partial weight gradients of a batch's chunks (mlp_ws_floats for Bcap rows)
  int Bcap = 0;
  int t = 0;
  double calib_b = 1.0;                     // calibration slope of the last training
  float* X = nullptr; float* Y = nullptr;   // features, target E_K - E_J
  int64_t n = 0, cap = 0;
  bool ready = false;
};
int64_t mlp_ws_floats(const int* dims, int B);   // workspace of mlp_backward for batches of at most B rows
void mlp_forward(const Mlp& m, const float* X, const int* idx, int B, hipStream_t st);
void mlp_backward(const Mlp& m, int B, hipStream_t st);
float mlp_loss(const Mlp& m, const float* t, const int* idx, int B, hipStream_t st);
void mlp_adam(Mlp& m, float lr, hipStream_t st);
void launch_features(const DevState& s, const int* idx, int n, float* X, int64_t dst0, hipStream_t st);
void launch_ek(const DevState& s, const int* idx, int n, double* ek, float* yout, int64_t dst0, hipStream_t st,
               const int* n_dev = nullptr);
void launch_predict(const DevState& s, const Mlp& m, const float* X, int n, double* S, hipStream_t st);
void launch_ej(const DevState& s, double* ej, hipStream_t st);
void launch_sub(double* a, const double* b, int n, hipStream_t st);  // a -= b
void launch_block_energy(const DevState& s, const double* center, double halfw, double* out, hipStream_t st);
void launch_step_inc(unsigned long long* step, hipStream_t st);
void launch_energy_cv(const DevState& s, const double* S, const double* ek, const float* pinv, double delta,
                      const double* soff_dev, const double* center, int nwr, double halfw, double* dres,
                      hipStream_t st);
// exact set of the control variate from the live list s.live / s.nlive (k_cv_select)
void launch_cv_select(const DevState& s, const unsigned char* risky, int m, uint64_t seed, uint64_t draw, int force,
                      int* tame, int* sel, int* nsel, float* pinv, hipStream_t st);
void launch_cv_stats(const DevState& s, const double* S, const double* EK, const double* EJ, const double* D,
                     const float* pinv, const int* sel, const int* nsel, hipStream_t st);
void launch_cv_offset(const DevState& s, double rate, hipStream_t st);
// buffers of the risk stratum's two radix sorts over W walkers
struct RiskSort {
  double* kin = nullptr; double* kout = nullptr;
  int* iin = nullptr; int* iout = nullptr;
  void* tmp = nullptr; size_t tmp_bytes = 0;
};
size_t risk_sort_bytes(int W);
void launch_risk_split(const DevState& s, const double* ej, double risk, RiskSort& rs, unsigned char* risky,
                       hipStream_t st);

// kernel launchers (afq_kernels.hip)
void launch_force_bias(const DevState& s, hipStream_t st);   // afq_force_bias.hip
// the workgroups of the FP64 force bias of a population: the 32 x 64 or the 64 x 64 tile, nz of them
// along K with m units each, np parts in the workspace, each a unit or (whole) a chunk
struct FbSplit { bool small, whole; int m, nz, np; double cost; };
FbOrder fb_order(int G, int64_t Ktot, int nslots);
void launch_fields(const DevState& s, const double* draws, uint64_t seed, uint64_t step, hipStream_t st);
void launch_vhs(const DevState& s, hipStream_t st);
void launch_propagate(const DevState& s, hipStream_t st);  // E psi, Taylor terms, E acc
bool prop_in_one(const DevState& s);   // launch_taylor is the whole propagation: the next and launch_expmul_post do nothing
void launch_expmul_pre(const DevState& s, hipStream_t st);
void launch_taylor(const DevState& s, hipStream_t st);
void launch_expmul_post(const DevState& s, hipStream_t st);
bool prop_fused_fits(const DevState& s);                              // k_prop_split handles N
bool prop64_fits(const DevState& s);                                  // k_prop64 handles N (afq_prop64.hip)
void launch_prop64(const DevState& s, double* dst, hipStream_t st);   // the fused FP64 propagation, result in dst
void launch_propagate_to(const DevState& s, double* dst, hipStream_t st);   // the whole propagation, result in dst
void launch_green(const DevState& s, bool all_walkers, hipStream_t st);
void launch_green_pre(const DevState& s, bool all_walkers, hipStream_t st);   // S, S^-1, log det S
void launch_theta_post(const DevState& s, hipStream_t st);                   // theta, e1 of the live walkers
// arguments of the Green's function kernels
struct GreenArgs {
  const double* psi; double* theta; double* logdet; double* e1; const double* weights; double* Sg;
  // fresh[w] = 1 when k_invert took walker w (its S^-1 in Sg is current); with
  // post = 1, k_theta takes the fresh walkers of nonzero weight only
  int* fresh = nullptr; int post = 0;
  // with tbh != nullptr, k_theta also writes theta split into Tb (hi tbh, lo tbl),
  // laid out as k_theta_split writes it
  unsigned short* tbh = nullptr; unsigned short* tbl = nullptr; int Np = 0, ctot = 0;
  const double* phi0; const double* phi1; const double* hphi0; const double* hphi1;
  int64_t ms, Ktot; int64_t det_off0, det_off1; int N, nslots, W; Slot s0, s1; int all;
};
constexpr int GN_MAX = 64;                              // electrons per slot at most
constexpr int SG_LD = 2 * GN_MAX;                       // doubles per row of an Sg matrix
constexpr int64_t SG_MAT = (int64_t)GN_MAX * SG_LD;     // doubles per (walker, slot)
void launch_overlap(const GreenArgs& a, hipStream_t st);   // afq_green.hip
void launch_theta(const GreenArgs& a, hipStream_t st);
void launch_weight(const DevState& s, double eshift, bool update_weights, hipStream_t st);
void launch_logO_from_logdet(const DevState& s, hipStream_t st);
void launch_qr(const DevState& s, hipStream_t st);
bool launch_qr_cols(const DevState& s, hipStream_t st);   // afq_qr.hip; false where it does not apply
// nsel_dev (nullable): the selection's length on the device; nsel is then the bound the
// grid is sized for
void launch_exchange(const DevState& s, const int* sel, int nsel, hipStream_t st, const int* nsel_dev = nullptr);
// the FP64 exchange kernel for slots of at least X64_NMIN electrons (afq_exchange64.hip):
// slots a and b (b of a's size; nz = 1: a alone), partials at xp
constexpr int X64_NMIN = 4;   // its tile holds (64 / n)^2 (vector, walker) pairs, one thread each at least
void launch_exchange64(const DevState& s, const int* sel, int nsel, const int* nsel_dev, double* xp, Slot a, Slot b, int nz,
                       hipStream_t st);
void launch_energy(const DevState& s, const int* sel, int nsel, double delta, hipStream_t st);
void launch_comb(DevState& s, double zeta, hipStream_t st);
void launch_live_list(const DevState& s, hipStream_t st);   // s.live / s.nlive: walkers of nonzero weight
void launch_step_stats(const DevState& s, hipStream_t st);  // SS_SUMW .. SS_NCAP
void launch_block_totals(const DevState& s, const double* center, int nwr, double halfw, bool clip,
                         double* st_out, hipStream_t st);   // SS_BW .. SS_NBAD
void launch_broadcast_det(const DevState& s, const double* src, hipStream_t st);
// 1-RDM accumulation: acc[e] += sum_w w Re theta[w][e] (e < Ktot), acc[Ktot] += sum_w w,
// over the walkers of nonzero weight; part holds rdm_part_doubles(s) doubles
int64_t rdm_part_doubles(const DevState& s);
void launch_rdm_accumulate(const DevState& s, double* part, double* acc, hipStream_t st);
inline int onebody_pitch(int N) { return (N + 31) / 32 * 32; }
void launch_v_split(const DevState& s, hipStream_t st);
void launch_rq8(const DevState& s, hipStream_t st);
void launch_d_split(const DevState& s, hipStream_t st);
void launch_copy_det0_to_det1(const DevState& s, double* dst, const double* src, hipStream_t st);

void launch_pack_chol(const double* L, double* Lp, int N, int G, int64_t T, bool round_f32, hipStream_t st);
void launch_rotate_chol(const double* L, const double* phi, double* R, int N, int n, int G, int64_t Ktot,
                        int64_t koff, hipStream_t st);
void launch_debug_gemm(const double* A, const double* B, double* C, int M, int N, int K, hipStream_t st);
void launch_debug_gemm_bf16(const double* A, const double* B, float* C, int M, int N, int K, int passes,
                            void* scratch, hipStream_t st);
void launch_copy_small(const double* a, double* b, int n, hipStream_t st);   // b may be pinned host memory
void launch_copy_calib(const double* a, double* b, int64_t n, hipStream_t st);
void launch_fill(double* p, int64_t n, double v, hipStream_t st);

void launch_rsplit(const DevState& s, hipStream_t st);
// pair-wise one-pass exchange: g-tiles per workgroup at most (the partials it keeps in
// LDS), and N padded to 32 at most for k_exchange_pw2 (theta of a walker in its LDS)
constexpr int PW_TMAX = 160;
constexpr int PW2_KMAX = 448;
// k_exchange_pw2<ceil(n/16), waves, x3> over (live walker, slot, chunk) workgroups of 4 or 8
// waves (afq_exchange_pw2.hip); x3: the three-pass split form (4 waves; rfl, tl the lo parts)
void launch_exchange_pw2(const unsigned short* rf, const unsigned short* rfl, int64_t rf_slot,
                         const unsigned short* th, const unsigned short* tl, const int* sel, const int* nsel_dev,
                         double* xp, int Np, int GE, int nw, int W, Slot a, Slot b, int ctot, int ngt_cap, int gt,
                         int tpc, int nz, int nchunk, int nb, int waves, bool x3, hipStream_t st);
// k_exchange_pw2x3<ceil(n/16)>: the three-pass form in the default register form
// (afq_exchange_pw2x3.hip), same arguments
void launch_exchange_pw2x3(const unsigned short* rf, const unsigned short* rfl, int64_t rf_slot,
                           const unsigned short* th, const unsigned short* tl, const int* sel, const int* nsel_dev,
                           double* xp, int Np, int GE, int nw, int W, Slot a, Slot b, int ctot, int ngt_cap, int gt,
                           int tpc, int nz, int nchunk, int nb, hipStream_t st);
// size of Rf in u16 (off: each slot's offset), 0 where k_exchange_pw2 does not apply
int64_t rfrag_elems(const DevState& s, int64_t* off);
void launch_rfrag(const DevState& s, hipStream_t st);
void launch_exchange_lp(const DevState& s, const int* sel, int nsel, int prec, hipStream_t st,
                        const int* nsel_dev = nullptr);
void launch_theta_split(const DevState& s, const int* sel, int nsel, hipStream_t st, const int* nsel_dev = nullptr);
void launch_force_bias_lp(const DevState& s, int prec, hipStream_t st);
void launch_lt_split(const DevState& s, hipStream_t st);
void launch_vhs_lp(const DevState& s, int prec, hipStream_t st);

int exchange_tile_g(int n);   // g-blocks per exchange tile for slot size n (0: unsupported)
int exchange_tile_w(int n);   // walkers per exchange tile

// Hands out 256-byte aligned pieces of one buffer; with base == nullptr it only sizes.
struct Carve {
  unsigned char* base;
  size_t off = 0;
  template <class T>
  T* take(size_t n) {
    off = (off + 255) & ~size_t(255);
    T* p = base ? reinterpret_cast<T*>(base + off) : nullptr;
    off += n * sizeof(T);
    return p;
  }
};

// The buffers of a temporary population of ndet walkers that the Green's function,
// force bias, exchange and energy kernels read or write, carved from c; every other
// walker buffer of t is null.
inline void carve_population(DevState& t, int ndet, Carve& c) {
  const int64_t n = ndet;
  t.psi = c.take<double>(2 * n * t.ms);
  t.theta = c.take<double>(2 * n * t.Ktot);
  t.fb = c.take<double>(2 * n * t.G);
  t.logO = c.take<double>(2 * n);
  t.e1 = c.take<double>(2 * n * t.nslots);
  t.logdet = c.take<double>(2 * n * t.nslots);
  t.weights = c.take<double>(n);
  t.Sg = c.take<double>(n * t.nslots * 64 * 128);
  t.fbw = t.Sg;
  t.fbw_doubles = n * t.nslots * 64 * 128;
  t.Xp = c.take<double>(2 * (int64_t)t.nslots * n * t.ngt_cap);
  t.eloc = c.take<double>(n);
  t.ho = c.take<double>(4 * n);
  t.live = c.take<int>(n);
  t.nlive = c.take<int>(1);
}

// a population of ndet walkers that shares s's Hamiltonian and trial and no walker buffer
// (carve_population sets those it needs); ge: Cholesky vectors in the energy
inline DevState temporary_population(const DevState& s, int ndet, int ge) {
  DevState t = s;
  t.factors = t.psi2 = t.theta2 = t.fb2 = t.logO2 = t.e12 = nullptr;
  t.fields = t.sft = t.P = t.t0 = t.t1 = t.accb = t.draws = t.cum = t.P2 = nullptr;
  t.idx = t.gfresh = nullptr;
  t.ncap = nullptr;
  t.Tb_hi = t.Tb_lo = nullptr;
  t.fbp = nullptr;
  t.fbp_rows = 0;
  t.tb_live = false;
  t.tb_post = false;
  t.d_step = nullptr;
  t.d_eshift = nullptr;
  t.d_zeta = nullptr;
  t.graph_mode = false;
  t.W = ndet;
  t.GE = ge;
  return t;
}
// (H, overlap) of its walkers into t.ho; FP64: this population is not the one the bf16 buffers cover
inline void launch_temporary(const DevState& t, hipStream_t st) {
  launch_fill(t.weights, t.W, 1.0, st);
  launch_green(t, true, st);
  launch_logO_from_logdet(t, st);
  launch_force_bias(t, st);
  if (t.GE > 0) launch_exchange(t, nullptr, t.W, st);
  launch_energy(t, nullptr, t.W, 0.0, st);
}

}  // namespace afq

// One context: one rank's walker population, the Hamiltonian and the trial on one GPU
// (the object behind the C ABI's afq_ctx handle).
struct afq_ctx {
  afq::DevState s;
  afq_params params{};
  hipStream_t stream = nullptr;
  std::string err;
  // a kept block for temporary populations, pinned memory for small results, and who uses them
  std::mutex tmp_mu, pin_mu;
  unsigned char* tmp = nullptr;
  size_t tmp_bytes = 0;
  double* pin = nullptr;
  bool prepped = false;
  bool have_walkers = false;
  // set by afq_set_weights: a walker it revives may carry a force bias older than its
  // orbitals (a step computes the force bias only for the walkers it leaves alive), so
  // the next reader of the force bias recomputes theta and the force bias first
  bool fb_stale = false;
  std::vector<double> h1, h1mod, chol;  // host copies (setup math)
  std::vector<double> h1d, h1modd, chold;  // down-spin copies with unrestricted integrals
  std::vector<double> phi[2];
  std::vector<float> dummy;
  // stage timing
  struct EvPair { hipEvent_t a, b; int stage; bool first; };   // first: a is not another pair's b
  std::vector<EvPair> pending;
  std::vector<hipEvent_t> pool;
  double stage_ms[afq::ST_COUNT] = {0};
  bool timing = true;
  // surrogate control variate (its running offset, counts and residual statistics live in
  // the device statistics s.stats)
  afq::Mlp mlp;
  int cv_minv = 16;
  double cv_risk = 0.05;
  int cv_kind = AFQ_SURR_MLP;
  int cv_prec = AFQ_PREC_BF16;   // precision of the AFQ_SURR_EXCHANGE level
  double cv_offset_rate = 0.1;
  double cv_fallback = 0.0;
  uint64_t cv_seed = 1;         // Philox key of the exact-set draws
  uint64_t cv_draw = 0;         // draws so far (the Philox counter)
  int cv_force = -1;            // >= 0: every block takes this position (test hook)
  bool cv_last_fallback = false;
  int64_t cv_nfallback = 0;
  double* cvS = nullptr;
  double* cvEK = nullptr;
  double* cvEJ = nullptr;
  float* cvPinv = nullptr;
  double* cvD = nullptr;        // clipped exact - surrogate energy of the exact set
  double* cvCenter = nullptr;   // clip centres, walker w uses cvCenter[w / cv_nwr] (null: no clipping)
  int cv_nwr = 1;
  double cv_halfw = 0.0;
  int* cvSel = nullptr;         // the exact set (device), its length in *cvNsel
  int* cvNsel = nullptr;
  int* cvTame = nullptr;        // live walkers outside the risk stratum (scratch of the draw)
  unsigned char* cvRisky = nullptr;
  afq::RiskSort rsort;
  float* cvX = nullptr;
  bool last_exact_all = false;
  bool last_measure_clipped = false;   // the last measurement's energies are clipped already
  // mixed-estimator 1-RDM: acc[e] = sum w Re theta[e] (e < Ktot), acc[Ktot] = sum w
  double* rdmAcc = nullptr;
  double* rdmPart = nullptr;

  // per-stage device timers (HIP events on the context's stream)
  hipEvent_t ev_get();
  void stage_begin(int st, EvPair& p);
  void stage_next(int st, EvPair& p);
  void stage_end(EvPair& p);
  void resolve();
};
