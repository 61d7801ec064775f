/*
 * vmc_afqmc.h -- C ABI of the MI355X phaseless-AFQMC walker step.
 *
 * One context (afq_ctx) holds one rank's whole walker population, the
 * Hamiltonian tensors and the trial on one GPU.  Every call is stream-ordered
 * on the context's HIP stream; a context is not re-entrant (one host thread at
 * a time).  All calls return AFQ_OK (0) or a nonzero status; the message of the
 * last failure is available from afq_last_error().  The library never calls
 * exit(); numeric failures of single walkers are reported through weights and
 * flags exactly as the reference does (weight factor 0).
 *
 * Data conventions (host buffers unless a name ends in _dev):
 *   - complex numbers are interleaved (re, im) doubles, i.e. the memory layout
 *     of std::complex<double> / double _Complex;
 *   - matrices are row-major unless stated otherwise;
 *   - walker determinants use the reference's serial layout
 *     (DQMC/DQMCWalker.cpp:251-290): for each walker, psi_up row-major
 *     norb x nalpha, then psi_dn row-major norb x nbeta (mat_size =
 *     norb*(nalpha+nbeta) complex numbers per walker).
 *
 * Reference interfaces replaced (paths relative to the sanshar/VMC tree):
 *   afq_create          Hamiltonian ctor + floattenCholesky + RHF/UHF left-trial
 *                       ctor with rotateCholesky  (DQMC/Hamiltonian.cpp:9-42,
 *                       52-133,179-220; DQMC/RHF.cpp:9-17; DQMC/UHF.cpp:9-21)
 *   afq_set_nchol_ene   Hamiltonian::setNcholEne (DQMC/Hamiltonian.cpp:45-48)
 *   afq_prep_prop       DQMCWalker::prepPropR (DQMC/DQMCWalker.cpp:32-103)
 *   afq_set_walkers     DQMCWalker::setDet(serial, overlap) (DQMC/DQMCWalker.cpp:251-269)
 *   afq_get_walkers     DQMCWalker::getDet (DQMC/DQMCWalker.cpp:272-290)
 *   afq_propagate       walker loop of calcMixedEstimatorLongProp with
 *                       DQMCWalker::propagatePhaselessRG
 *                       (DQMC/MixedEstimator.cpp:461-468; DQMC/DQMCWalker.cpp:441-503)
 *   afq_orthogonalize   DQMCWalker::orthogonalize loop (DQMC/MixedEstimator.cpp:478-480;
 *                       DQMC/DQMCWalker.cpp:295-326)
 *   afq_measure         DQMCWalker::hamAndOverlap loop with the E_L clip
 *                       (DQMC/MixedEstimator.cpp:489-533; DQMC/RHF.cpp:104-131;
 *                       DQMC/UHF.cpp:75-106)
 *   afq_force_bias      DQMCWalker::forceBias (DQMC/DQMCWalker.cpp:569-576;
 *                       DQMC/RHF.cpp:42-61; DQMC/UHF.cpp:45-65)
 *   afq_overlap         DQMCWalker::overlap (DQMC/DQMCWalker.cpp:559-566)
 *   afq_comb            reconfiguration (DQMC/MixedEstimator.cpp:559-635)
 *   afq_rdm_accumulate  DQMCWalker::oneRDM loop of the mixed-estimator 1-RDM
 *                       (DQMC/MixedEstimator.cpp:492-510; DQMC/DQMCWalker.cpp:579-589;
 *                       DQMC/RHF.cpp:64-67; DQMC/UHF.cpp:68-72)
 *   afq_get_one_rdm     oneRDM / cumulativeWeight as writeOneRDM writes them
 *                       (DQMC/MixedEstimator.cpp:52-112)
 *   afq_run_long_prop   calcMixedEstimatorLongProp (DQMC/MixedEstimator.cpp:309-699)
 */
#ifndef VMC_AFQMC_H
#define VMC_AFQMC_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define AFQ_ABI_VERSION 1

/* status codes */
#define AFQ_OK 0
#define AFQ_ERR_ARG 1          /* bad argument / shape */
#define AFQ_ERR_DEVICE 2       /* HIP runtime failure */
#define AFQ_ERR_UNSUPPORTED 3  /* shape or mode this build does not support */
#define AFQ_ERR_STATE 4        /* call out of order (e.g. propagate before prep_prop) */
#define AFQ_ERR_NUMERIC 5      /* NaN/Inf local energy (reference exits, we report) */

/* arithmetic used by a stage (afq_params.prec_*) */
#define AFQ_PREC_FP64 0    /* plain double precision                          */
#define AFQ_PREC_FP32 1    /* float operands, float accumulation              */
#define AFQ_PREC_BF16X3 2  /* bf16 hi/lo split, 3 MFMA passes, fp32 accumulate */
#define AFQ_PREC_BF16 3    /* one bf16 pass, fp32 accumulate                  */
#define AFQ_PREC_FP8 4     /* e4m3 with per-Cholesky-vector scale + fp32 residual */

/* local-energy evaluation (afq_measure mode) */
#define AFQ_ENERGY_EXACT 0      /* exact E_L on every live walker                   */
#define AFQ_ENERGY_SURROGATE 1  /* surrogate exchange on all + exact on a subset, */
                                /* two-level control variate (needs a surrogate)    */

/* Hamiltonian in the fields of the reference's FCIDUMP_chol
 * (utils/integral.cpp:589-661, scripts/QMCUtils.py:1067-1075). */
typedef struct afq_ham {
  int32_t norb;        /* N                                  */
  int32_t nalpha;      /* electrons of spin up               */
  int32_t nbeta;       /* electrons of spin down             */
  int32_t nchol;       /* G, number of Cholesky vectors       */
  double ecore;        /* energy_core                        */
  const double* h1;     /* hcore, N x N                      */
  const double* h1_mod; /* hcore_mod = hcore - 1/2 sum_g L_g L_g, N x N */
  const double* chol;   /* G x N x N, row g = vec(L_g), each L_g symmetric */
  /* Unrestricted integrals (intType "u": /hcore_up, /hcore_dn, /hcore_mod_up,
   * /hcore_mod_dn, /chol_up, /chol_dn, utils/integral.cpp:664-741): with h1_dn,
   * h1_mod_dn and chol_dn non-null, h1, h1_mod and chol are the up-spin ones and
   * the walk is propagatePhaselessU (DQMC/DQMCWalker.cpp:106-187, 506-554); this
   * needs a UHF trial, UHF walkers and FP64 VHS and propagation.  All three null:
   * restricted integrals. */
  const double* h1_dn;
  const double* h1_mod_dn;
  const double* chol_dn;
} afq_ham;

/* Left trial (RHF or UHF, DQMC/RHF.h, DQMC/UHF.h).  Orbitals are real. */
typedef struct afq_trial {
  int32_t rhf;          /* 1: RHF (phi_dn ignored, nalpha == nbeta required) */
  const double* phi_up; /* N x nalpha, row-major                            */
  const double* phi_dn; /* N x nbeta, row-major                             */
} afq_trial;

typedef struct afq_params {
  int32_t nwalk;       /* walkers in this context                                  */
  int32_t walker_rhf;  /* DQMCWalker::rhfQ: one determinant shared by both spins   */
                       /* (requires nalpha == nbeta; executables/DQMC.cpp:74-82)    */
  int32_t ref_compat;  /* 1: round L and fields to float in the VHS and mean-field */
                       /* shifts like the reference (DQMC/DQMCWalker.cpp:73-84,454) */
  int32_t prec_fb;     /* force bias arithmetic  (AFQ_PREC_*)                     */
  int32_t prec_vhs;    /* VHS arithmetic                                           */
  int32_t prec_exchange; /* exchange contraction arithmetic                      */
  int32_t device;      /* HIP device ordinal                                       */
  double weight_cap;   /* <= 0: max(100, nwalk/10) (DQMC/MixedEstimator.cpp:452-454) */
} afq_params;

typedef struct afq_ctx afq_ctx;

/* Message of the last failure on ctx (or of the last failed afq_create when
 * ctx is NULL).  Valid until the next call on the same context. */
const char* afq_last_error(const afq_ctx* ctx);

/* Library / ABI version; also forces the shared object to load. */
int afq_version(void);

/* Create a context: uploads h1, h1_mod, L_g (FP64), the packed lower-triangle
 * L (floattenCholesky layout) and the half-rotated Cholesky R_{s,g} = Phi_s^T L_g
 * of the left trial.  Allocates the walker population (all weights 0 until
 * afq_set_walkers). */
int afq_create(const afq_ham* ham, const afq_trial* left, const afq_params* params,
               afq_ctx** out);
int afq_destroy(afq_ctx* ctx);

/* Change the arithmetic of the stages on an existing context (the walker
 * population is kept).  Each of prec_fb (force bias), prec_vhs (VHS) and
 * prec_exchange (exchange contraction) is AFQ_PREC_FP64, AFQ_PREC_BF16X3 (bf16
 * hi/lo split, three MFMA passes, FP32 accumulation: about FP32 accuracy) or
 * AFQ_PREC_BF16 (one pass).  Overlaps, Green's functions, the propagation,
 * weights and QR stay FP64.  ref_compat contexts need prec_vhs = AFQ_PREC_FP64. */
int afq_set_precision(afq_ctx* ctx, int32_t prec_fb, int32_t prec_vhs, int32_t prec_exchange);
/* Arithmetic of the five Taylor products V t of the propagation: AFQ_PREC_FP64
 * (default) or AFQ_PREC_BF16X3 (split-BF16 MFMA, FP32 accumulation; V and t stay
 * FP64 in memory and the series is accumulated in FP64). */
int afq_set_prop_precision(afq_ctx* ctx, int32_t prec_prop);

/* Number of Cholesky vectors used by the local energy (default nchol). */
int afq_set_nchol_ene(afq_ctx* ctx, int32_t nchol_ene);

/* Mean-field background subtraction and one-body propagator.
 * ref_up/ref_dn: reference determinant (N x nalpha / N x nbeta, row-major)
 * used for Gref = ref (ref^T ref)^-1 ref^T unless rdm_up/rdm_dn (N x N) are
 * given (the spinRDM.0.0.txt path).  ene0 is accepted for interface parity;
 * the phaseless propagator constant does not depend on it. */
int afq_prep_prop(afq_ctx* ctx, const double* ref_up, const double* ref_dn,
                  const double* rdm_up, const double* rdm_dn, double dt, double ene0);

/* Walker population I/O in the serial layout.  overlaps (complex, nwalk) may be
 * NULL on set: the trial overlap is then computed (DQMCWalker::overlap).
 * weights may be NULL on set (all 1).  Any output pointer may be NULL on get. */
int afq_set_walkers(afq_ctx* ctx, const double* dets, const double* overlaps,
                    const double* weights);
int afq_get_walkers(afq_ctx* ctx, double* dets, double* overlaps, double* weights);
int afq_get_weights(afq_ctx* ctx, double* weights);
int afq_set_weights(afq_ctx* ctx, const double* weights);
/* Every walker a copy of one determinant (det: one walker's serial block) with the given
 * weight, as the reference copies its walker prototype into the population
 * (DQMC/MixedEstimator.cpp:399-410); the copy happens on the device.  overlap (one
 * complex, nullable): the trial overlap, computed when NULL. */
int afq_set_walkers_uniform(afq_ctx* ctx, const double* det, const double* overlap, double weight);

/* One phaseless step of the whole population.  draws: nwalk x nchol standard
 * normals, row w used only if walker w is alive (weight > 1e-8), or NULL to draw
 * on the device from (seed, walker slot, step) with a counter-based generator.
 * Applies weight *= factor for live walkers and the weight cap; returns the
 * per-walker factors in factors (nullable) and the number of walkers zeroed by
 * the cap in n_capped (nullable).  eshift as in DQMC/MixedEstimator.cpp:475. */
int afq_propagate(afq_ctx* ctx, const double* draws, uint64_t seed, uint64_t step,
                  double eshift, double* factors, int64_t* n_capped);

/* Householder re-orthonormalisation of every walker of nonzero weight (Eigen's sign
 * convention, R_kk = -sign(Re x_0) |x|), trialOverlap /= prod diag R.  A walker of
 * weight zero is left as it is: it is neither propagated nor measured before the comb
 * replaces it. */
int afq_orthogonalize(afq_ctx* ctx);

/* Local energies of every walker with weight != 0; dead walkers get eloc 0 and
 * E*O = 0 (their exchange is not computed, as the reference computes no local
 * energy for them, DQMC/MixedEstimator.cpp:531).
 * mode AFQ_ENERGY_EXACT: eloc[w] = Re(E*O/O) + delta.  ham_ovlp (nullable):
 * per walker {E*O, O} as two complex numbers (hamAndOverlap).  The exact mode does
 * not clip (the caller clips, DQMC/MixedEstimator.cpp:525-530); the surrogate mode
 * clips inside its estimate when afq_set_energy_clip set a clip. */
int afq_measure(afq_ctx* ctx, int32_t mode, double delta, double* eloc, double* ham_ovlp);

/* E_L of arbitrary determinants against the left trial (init-time helper used
 * for the reference energy and the Cholesky truncation search,
 * DQMC/MixedEstimator.cpp:352-384).  dets: ndet determinants in serial layout;
 * out: ndet x {E*O, O} complex.  FP64 results of a determinant or a walker (these, the
 * force bias, the exact energies) do not depend on how many others one call takes. */
int afq_ham_and_overlap(afq_ctx* ctx, const double* dets, int32_t ndet,
                        int32_t nchol_ene, double* out);

/* E_L of arbitrary determinants with no device allocation: afq_ham_and_overlap on
 * device buffers.  No counterpart in the reference; for callers that cannot allocate
 * device memory (code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc).  dets_dev: ndet determinants in the serial layout (device);
 * out_dev: ndet x {E*O, O} complex (device).  The temporary population lives in a
 * device array of AFQ_NOALLOC_SCRATCH_BYTES that each GPU holds until the process
 * ends; a call that needs more (about 48 determinants at N=300, 60+60, G=1200)
 * returns AFQ_ERR_ARG.  Stream-ordered on the context's stream and returns without
 * waiting (afq_sync before reading out_dev).  Every call on one GPU shares that
 * GPU's array, which keeps the last call's contents: calls that overlap on one GPU
 * race. */
#define AFQ_NOALLOC_SCRATCH_BYTES (64ull << 20)
int afq_ham_and_overlap_dev(afq_ctx* ctx, const double* dets_dev, int32_t ndet, int32_t nchol_ene,
                            double* out_dev);

/* Parity hooks: force bias (nwalk x nchol complex) and trial overlaps of the
 * current population, computed from the current determinants (walkers given weight
 * again by afq_set_weights get theta and the force bias recomputed first).  The force
 * bias is kept for walkers of nonzero weight only; a dead walker's entries are stale. */
int afq_force_bias(afq_ctx* ctx, double* fb);
int afq_overlap(afq_ctx* ctx, double* overlaps);

/* ---------------------------------------------------------------- population statistics
 * The numbers calcMixedEstimatorLongProp's population control reads
 * (DQMC/MixedEstimator.cpp:461-475, 513-538, 595-622), kept on the device so that a step
 * needs one small copy to the host (afq_get_step_stats) instead of per-walker arrays:
 *   - afq_propagate records the sum of the weights after its weight update (in walker
 *     order, as the reference's loop adds them), the walkers it propagated (weight >
 *     1e-8 at its start), the walkers of nonzero weight after it and the walkers capped;
 *   - afq_block_totals records the block totals of the last afq_measure: every live
 *     walker's local energy clipped to its clip centre -+ halfwidth (when a clip is set
 *     and the measurement did not clip already; DQMC/MixedEstimator.cpp:525-530), sum w,
 *     sum w E_L in walker order, the variance of the weighted mean and the counts;
 *   - a surrogate measurement records its exact-set size and residual statistics;
 *   - afq_comb records the total weight it distributed. */
typedef struct afq_step_stats {
  double total_weight;    /* sum of all weights after the last afq_propagate                  */
  int64_t n_propagated;   /* walkers it propagated (weight > 1e-8 at its start)              */
  int64_t n_live;         /* walkers of nonzero weight after it                               */
  int64_t n_capped;       /* walkers its weight cap zeroed                                    */
  double block_weight;    /* last afq_block_totals: sum w over the live walkers               */
  double block_wsum;      /*   sum w E_L (clipped), walker order                              */
  double block_var;       /*   sum w^2 (E_L - E)^2 / (sum w)^2, E = block_wsum / block_weight */
  int64_t n_measured;     /*   live walkers (each has a local energy)                         */
  int64_t n_clipped;      /*   local energies the clip moved                                  */
  int64_t n_nonfinite;    /*   NaN / Inf local energies of live walkers                        */
  int64_t n_exact;        /* last surrogate measurement: walkers measured exactly             */
  double cv_rms;          /*   residual RMS of its random part (Ha)                           */
  double cv_var_sub;      /*   subset-sampling variance of the weighted mean energy (Ha^2)    */
  double cv_mean_resid;   /*   mean residual (Ha)                                             */
  int32_t cv_fallback;    /*   1: every walker was measured exactly instead                   */
  double comb_total;      /* last afq_comb: the total weight                                  */
} afq_step_stats;
/* Clip centres for the local energies (the running averages of the reference's ranks):
 * walker w uses centers[w / (nwalk / ncenters)], ncenters must divide nwalk; the
 * surrogate measurement clips with them inside its estimate (as afq_set_energy_clip)
 * and afq_block_totals clips exact energies with them.  centers == NULL or
 * halfwidth <= 0: no clip. */
int afq_set_clip_centers(afq_ctx* ctx, const double* centers, int32_t ncenters, double halfwidth);
int afq_block_totals(afq_ctx* ctx);
/* waits for the context's stream, then one small copy */
int afq_get_step_stats(afq_ctx* ctx, afq_step_stats* out);

/* Comb reconfiguration with the uniform zeta (DQMC/MixedEstimator.cpp:595-622):
 * new walker w is old walker lower_bound(cum, (w+zeta)/W * sum). Sets every
 * weight to sum/W.  total_weight (nullable) receives sum. */
int afq_comb(afq_ctx* ctx, double zeta, double* total_weight);

/* Mixed-estimator one-body density matrix (DQMC/MixedEstimator.cpp:492-510).
 * afq_rdm_accumulate adds one measurement: every walker of nonzero weight w
 * contributes w Re(G_s^T) per spin slot s, G_s = psi_s (Phi_s^T psi_s)^-1 Phi_s^T
 * (RHF::oneRDM DQMC/RHF.cpp:64-67, UHF::oneRDM DQMC/UHF.cpp:68-72), from the
 * Green's function of the current determinants, and w to the cumulative weight.
 * afq_get_one_rdm returns the weighted average (the reference keeps it as a
 * running average, oneRDM = (oneRDM cw + w sample) / (cw + w)) and the cumulative
 * weight: spin_summed = 1 gives one N x N row-major matrix, both spins added
 * (RHF::oneRDM); spin_summed = 0 gives two, up then down (UHF::oneRDM).  With
 * no accumulation yet both are zero.  afq_rdm_reset clears the accumulator. */
int afq_rdm_reset(afq_ctx* ctx);
int afq_rdm_accumulate(afq_ctx* ctx);
int afq_get_one_rdm(afq_ctx* ctx, int32_t spin_summed, double* rdm, double* cumulative_weight);

/* Per-stage device time (ms) accumulated since the last reset, AFQ_NSTAGES
 * entries in the order force_bias, fields, vhs, one-body (E psi), green, weight,
 * ortho, exchange, comb, taylor (the five V t products; the whole propagation where
 * one kernel does it, and one-body is then 0), exchange_lp (the reduced-precision
 * exchange of the AFQ_SURR_EXCHANGE surrogate). */
#define AFQ_NSTAGES 11
int afq_stage_times(afq_ctx* ctx, double* ms, int32_t reset);

/* ---------------------------------------------------------------- surrogate
 * Exchange-energy surrogate (no counterpart in the reference): a GELU MLP
 * F -> hidden -> hidden -> hidden -> 1, F = nchol + 2 norb, fed Re fb_g and
 * Re diag G_up/dn, trained on the GPU (BF16 MFMA GEMMs, FP32 accumulation,
 * FP32 master weights, Adam, MSE) on (walker features, exact E_K - E_J) pairs
 * that afq_surrogate_collect takes from exact measurements.  The risk stratum,
 * the fraction risk_frac of live walkers whose Coulomb energy E_J lies farthest
 * from the median, is always evaluated exactly (and is left out of training).
 * afq_measure with AFQ_ENERGY_SURROGATE then evaluates E_L = E_1 - S(x) on every
 * walker plus pinv (S - (E_K - E_J)) on the exact set: the risk stratum
 * (pinv = 1) and one walker drawn from each block of subset_inv remaining live
 * walkers (pinv = block size), an unbiased Horvitz-Thompson estimate of every
 * walker's exact E_L.  Every walker is measured exactly instead when the random
 * part's residual RMS exceeds fallback_rms (0: never). */
int afq_surrogate_init(afq_ctx* ctx, int32_t hidden, uint64_t seed, int64_t capacity);
int afq_surrogate_collect(afq_ctx* ctx, int64_t* total);
/* append n external (features X[n x F], target Y[n]) pairs to the training set */
int afq_surrogate_load(afq_ctx* ctx, const float* X, const float* Y, int64_t n, int64_t* total);
/* Adam on the first nine tenths of the samples (collection order); the last tenth
 * validates.  The weights of the epoch with the lowest validation RMSE are kept and
 * the output is calibrated on the validation set to a + b * net, b = max(0,
 * cov(y, net) / var(net)), so a network that predicts nothing becomes a constant. */
int afq_surrogate_train(afq_ctx* ctx, int32_t epochs, int32_t batch, double lr, uint64_t seed,
                        double* train_rmse, double* valid_rmse);
int afq_surrogate_predict(afq_ctx* ctx, double* pred);
/* flattened parameters: W0 b0 W1 b1 W2 b2 W3 b3 (W_l row-major in x out), mu[F], sd[F], t_mu, t_sd */
int afq_surrogate_params(afq_ctx* ctx, float* buf, int64_t nbuf, int32_t set);
/* one forward + backward pass on raw features X (B x F) and targets t (B): gradients of
 * 1/2 mean((y - (t - t_mu)/t_sd)^2) in the order of afq_surrogate_params (weights/biases only) */
int afq_surrogate_grad(afq_ctx* ctx, const float* X, const float* t, int32_t B, float* grads, double* loss);
int afq_set_cv(afq_ctx* ctx, int32_t subset_inv, double risk_frac, double fallback_rms, uint64_t seed);
/* per-walker one-body energy sum_s m_s tr(G_s h1) and exchange energy E_K (real
 * parts) of the last exact measurement of every walker; a walker of weight zero gets
 * E_K = 0 (the measurement computes no exchange for it).  Needs an exact measurement
 * after the last change of walkers or weights (afq_set_walkers, afq_set_weights,
 * afq_propagate, afq_comb). */
int afq_energy_parts(afq_ctx* ctx, double* e1, double* ek);
/* surrogate input features of every walker (nwalk x (nchol + 2 norb), float) */
int afq_surrogate_features(afq_ctx* ctx, float* X);
/* Surrogate of the control variate (AFQ_ENERGY_SURROGATE):
 *   AFQ_SURR_MLP       the trained network (default);
 *   AFQ_SURR_EXCHANGE  the exchange contraction itself in reduced precision `prec`
 *                      (AFQ_PREC_BF16 or AFQ_PREC_BF16X3) on every walker; the exact
 *                      set is then evaluated in the context's exchange precision. */
#define AFQ_SURR_MLP 0
#define AFQ_SURR_EXCHANGE 1
int afq_set_surrogate_kind(afq_ctx* ctx, int32_t kind, int32_t prec);
/* Clip applied inside the control-variate estimate: the surrogate-level and the
 * exact energy of walker w are both clipped to center[w] -+ halfwidth before the
 * Horvitz-Thompson correction (DQMC/MixedEstimator.cpp:525-530 clips every local
 * energy to the running average -+ sqrt(2/dt) on the host; clipping the corrected
 * estimate instead would bias it).  center == NULL or halfwidth <= 0: no clip. */
int afq_set_energy_clip(afq_ctx* ctx, const double* center, double halfwidth);
/* {exact-set size, residual RMS of its random part (Ha), fallback used, subset-sampling
 *  variance estimate of the weighted mean energy (Ha^2), mean residual, cumulative
 *  fallbacks} of the last surrogate measurement */
int afq_cv_stats(afq_ctx* ctx, double* out6);
/* Test hook of the control variate's exact set: position >= 0 makes every block take
 * its walker at position (position mod block size) instead of a uniform draw; averaging
 * the estimate over position = 0 .. subset_inv - 1 then gives every walker's exact
 * (clipped) energy when subset_inv divides the number of live walkers outside the risk
 * stratum.  position < 0: uniform draws (the default). */
int afq_debug_cv_force_position(afq_ctx* ctx, int32_t position);

/* ---------------------------------------------------------------- tuning
 * Propagation-kernel autotuner (no counterpart in the reference): times the kernel
 * variants of the context's whole propagation E (sum V^k/k!) E in its precision on its
 * current walkers (without changing them) and keeps the fastest.  FP64: 1 = 64 x 128 real
 * tiles, 2 = 128 x 128 complex tiles, and, where it applies (N <= 384), the fused kernel.
 * Split BF16: 1 = 128-orbital and 2 = 160-orbital row tiles with the one-body factors and
 * each Taylor step as separate kernels, 3 = one fused kernel per block of columns (N <= 384
 * only).  choice (nullable) receives the variant; in FP64 it names the better of 1 and 2
 * also where the fused kernel is kept, and handing it to afq_set_taylor_variant then turns
 * that kernel off (0 keeps it on).  ms3 (nullable, 3 entries): the times in ms per
 * propagation (0 for a variant not tried, and for the third in FP64). */
int afq_autotune(afq_ctx* ctx, int32_t* choice, double* ms3);
/* 0: by shape (default: the fused kernel where it applies), 1, 2 or 3: the variants
 * named at afq_autotune (3 falls back to the shape rule where N > 384 or in FP64, whose
 * rule is the fused kernel up to N = 384) */
int afq_set_taylor_variant(afq_ctx* ctx, int32_t variant);
/* One-pass BF16 exchange kernel (no counterpart in the reference): 0 by shape (default:
 * the pair-wise kernel with R in fragment order and two waves per SIMD wherever every
 * slot has at most 64 electrons and N <= 448, else the earlier pair-wise kernel wherever
 * N <= 512, else the tiled kernel), 1 the tiled kernel (128 x 128 output tiles, pair
 * sums through LDS), 2 the earlier pair-wise kernel, 3 the fragment-order kernel with one
 * wave per SIMD, 4 that kernel with two waves per SIMD (as 0 where it applies). */
int afq_set_exchange_variant(afq_ctx* ctx, int32_t variant);
/* Chunks of the Cholesky vectors the pair-wise one-pass exchange splits each (walker,
 * slot) into, one workgroup each (no counterpart in the reference; 0: by shape).  All
 * walkers take the chunks in the same order, so more chunks keep the rotated Cholesky
 * rows the resident workgroups read within the L2 of their XCD. */
int afq_set_exchange_chunks(afq_ctx* ctx, int32_t chunks);
/* FP64 exchange kernel (no counterpart in the reference): 0 (default) 64-row x 64-complex-
 * column tiles whose operands go straight from memory to registers, for slots of at least
 * 4 electrons (below: as 2, with 8 waves); 128 x 128 tiles through LDS: 1 the element-loader
 * engine (two barriers per stage), 2 the pointer-loader engine (double-buffered stages, 4 waves). */
int afq_set_exchange64_variant(afq_ctx* ctx, int32_t variant);
/* Split-BF16 VHS tile (no counterpart in the reference): 0 128 (walker, component) rows
 * by one 16 x 8 block of V, 64-deep single-buffered stages; 1 256 rows, eight waves,
 * 32-deep double-buffered stages; 2 128 rows, 32-deep double-buffered; 3 (default) and 4
 * as 0 and 2, with the split output of the blocks below the diagonal staged through LDS
 * and written as 16-byte runs (the others store each element's hi and lo at both
 * symmetric positions with 2-byte writes). */
int afq_set_vhs_tile(afq_ctx* ctx, int32_t tile);
/* Three-pass split-BF16 exchange (AFQ_PREC_BF16X3, the control variate's exact level; no
 * counterpart in the reference): 0 (default) the pair-wise kernel with R in fragment
 * order (k_exchange_pw2x3) wherever the largest slot has 13 to 64 electrons and N <= 448,
 * else the tiled kernel; 1 the tiled kernel; 2 as 0 with the pair-wise kernel compiled
 * with its MFMA accumulators in VGPRs (the one-pass kernel's register form; 11% slower). */
int afq_set_exchange3_variant(afq_ctx* ctx, int32_t variant);
/* Split-BF16 force bias (no counterpart in the reference): 0 (default) one workgroup per
 * output tile and slot, the two slots' FP32 sums added in FP64 by a second kernel (twice
 * the workgroups, for an even fill of the GPU); 1 one workgroup per output tile over both
 * slots (FP32 sum). */
int afq_set_force_bias_variant(afq_ctx* ctx, int32_t variant);

/* ---------------------------------------------------------------- batched systems
 * Many independent populations of different sizes on one GPU (no counterpart in the
 * reference, which runs one system per process).  afq_batch_create makes one
 * context per system; prepare each through afq_batch_context (afq_prep_prop,
 * afq_set_walkers, precision, afq_autotune), then afq_batch_capture records one step
 * of every system -- propagation, QR when step % ortho_steps == 0, exact energies of
 * every walker, block totals with the clip, comb -- into a hipGraph with one branch
 * per system.  afq_batch_step replays it: per system the energy shift, comb uniform
 * and clip centre go in, {sum w, sum w clip(E_L)} comes out (one copy each way).
 * The captured step is grouped by default: the systems' launches of each stage that
 * run the same kernel become one launch over all of their workgroups, so a step is one
 * launch per stage and kernel for all systems together.  afq_batch_set_lanes(b, k)
 * before the capture deals the systems over k streams grouped this way (k = 1 is the
 * default), or, with k = 0, records one graph branch per system instead.
 * The device RNG draws Philox(seed + 7919 i, step, walker) for system i, the step
 * counter starting at first_step.  After the capture the systems' buffers must not
 * be re-pointed: drive them only through afq_batch_step (or capture again). */
typedef struct afq_batch afq_batch;
int afq_batch_create(int32_t nsys, const afq_ham* hams, const afq_trial* trials, const afq_params* params,
                     afq_batch** out);
int afq_batch_destroy(afq_batch* b);
int afq_batch_context(afq_batch* b, int32_t i, afq_ctx** ctx);
/* lanes 1 .. 8: grouped launches on that many streams (default 1); 0: one graph branch
 * per system.  Takes effect at the next afq_batch_capture. */
int afq_batch_set_lanes(afq_batch* b, int32_t lanes);
int afq_batch_capture(afq_batch* b, uint64_t seed, int32_t ortho_steps, double clip_halfwidth,
                      uint64_t first_step);
/* Kernel launches in one captured step (qr = 1: the step with QR), -1 for the branch
 * form. */
int afq_batch_launches(afq_batch* b, int32_t qr, int32_t* launches);
/* graph = 0 issues the same kernels without the graph (for comparison) */
int afq_batch_step(afq_batch* b, int64_t step, const double* eshift, const double* zeta, const double* center,
                   int32_t graph, double* totals);
/* Per system, from the last afq_batch_step: the walkers its propagation took (weight
 * > 1e-8 at the step's start, the gate of DQMC/MixedEstimator.cpp:461-468) and the
 * walkers of nonzero weight that the measurement saw (before the comb). */
int afq_batch_counts(afq_batch* b, int64_t* propagated, int64_t* live);

/* ---------------------------------------------------------------- driver
 * calcMixedEstimatorLongProp (DQMC/MixedEstimator.cpp:309-699) on one GPU.
 * nranks virtual ranks of nwalk walkers each reproduce an `mpirun -np nranks`
 * run: rank r owns walkers [r*nwalk, (r+1)*nwalk) and, in replay mode, draws
 * from std::mt19937(seed + r) with one std::normal_distribution per walker slot
 * (executables/DQMC.cpp:58, DQMC/DQMCWalker.h:18); dead walkers draw nothing;
 * the comb's uniform comes from rank 0's generator. */
#define AFQ_RNG_REPLAY 0   /* the reference's libstdc++ stream, drawn on the host */
#define AFQ_RNG_DEVICE 1   /* counter-based Philox4x32-10 normals drawn on the GPU */

typedef struct afq_run_params {
  int64_t seed;
  double dt;
  int32_t nsteps;        /* steps per energy evaluation / reconfiguration     */
  int32_t nsweeps;       /* stochasticIter: number of blocks (samples lines)  */
  int32_t ortho_steps;
  int32_t burn_iter;
  int32_t nwalk;         /* per virtual rank                                  */
  int32_t nranks;
  int32_t walker_rhf;
  int32_t ref_compat;
  double cholesky_threshold;
  double ene0_guess;     /* 1e10: use the reference energy                   */
  double weight_cap;     /* <= 0: default                                     */
  int32_t max_steps;     /* > 0: stop after this many steps                   */
  int32_t rng_mode;      /* AFQ_RNG_REPLAY | AFQ_RNG_DEVICE                   */
  int32_t warmup_steps;  /* steps excluded from the timed region              */
  int32_t prec_fb, prec_vhs, prec_exchange;
  int32_t energy_mode;   /* AFQ_ENERGY_*                                      */
  int32_t device;
  /* surrogate control variate (energy_mode == AFQ_ENERGY_SURROGATE): the first
   * surrogate_train_steps steps measure exactly (FP64) and collect (features,
   * E_K - E_J) pairs, then the MLP is trained and the control variate takes over
   * (AFQ_SURR_MLP; the AFQ_SURR_EXCHANGE surrogate needs no training) */
  int32_t surrogate_train_steps;
  int32_t surrogate_hidden;
  int32_t surrogate_epochs;
  int32_t subset_inv;    /* exact E_L on a 1/subset_inv stratified subset     */
  double fallback_rms;   /* exact fallback when the subset residual RMS exceeds this (0: never) */
  double risk_frac;      /* fraction of live walkers always measured exactly  */
  int32_t shadow_exact;  /* 1: after each surrogate measurement also measure every walker
                          * exactly in FP64 (excluded from the timings) and report the
                          * difference of the two block energies on identical walkers */
  int32_t surrogate_kind; /* AFQ_SURR_MLP (trained first) | AFQ_SURR_EXCHANGE (no training) */
  int32_t surrogate_prec; /* precision of the AFQ_SURR_EXCHANGE level                      */
  int32_t prec_prop;      /* Taylor products (afq_set_prop_precision)                       */
  double* one_rdm_out;    /* non-null: receives the mixed-estimator 1-RDM, accumulated at every
                           * measurement with step dt > 10 and step > burn_iter nsteps
                           * (DQMC/MixedEstimator.cpp:492-510): N x N spin-summed for an RHF
                           * trial (RHF::oneRDM), 2 x N x N up then down for a UHF trial
                           * (UHF::oneRDM); its cumulative weight is one_rdm_weight          */
  const double* rdm_background; /* non-null: 2 x N x N (up, down) background density for the
                           * mean-field shifts in place of the reference determinant's, as
                           * prepPropR reads spinRDM.0.0.txt (DQMC/DQMCWalker.cpp:42-58)      */
  int32_t restart_every;  /* > 0: before steps 1 + k restart_every (k >= 1) every walker is reset
                           * to the initial determinant with weight 1, outside the timings (a
                           * benchmark aid that keeps a population stepping whose weights would
                           * otherwise fall below the propagation threshold for good); the
                           * energy estimates and shifts carry on.  0: never.                 */
} afq_run_params;

typedef struct afq_run_result {
  double ref_energy;
  int32_t nchol_ene;
  double delta;
  int64_t n_large_deviations;
  double prop_time, ene_time;  /* host wall seconds, as DQMC/MixedEstimator.cpp:664-676 */
  int64_t timed_steps;
  double timed_wall_s;         /* wall seconds of the steps after warmup_steps     */
  double stage_ms[AFQ_NSTAGES]; /* device time per stage (afq_stage_times order)    */
  double train_rmse, valid_rmse; /* surrogate fit (Ha)                             */
  double cv_var_sub;           /* mean subset-sampling variance of the block energy */
  double cv_rms;               /* mean residual RMS of the exact subset (Ha)        */
  int64_t cv_fallbacks;
  int64_t train_samples;
  double est_var;              /* mean over timed blocks of sum w^2 (E_L - E)^2 / (sum w)^2 (Ha^2) */
  int64_t shadow_n;            /* blocks with a shadow exact measurement                 */
  double shadow_shift;         /* mean of (surrogate - exact FP64) block energy (Ha)     */
  double shadow_var;           /* variance of that difference over the blocks (Ha^2)    */
  double shadow_est_var;       /* est_var of the exact FP64 energies of the same blocks */
  double shadow_wall_s;        /* wall seconds spent in shadow measurements (not timed) */
  double live_frac;            /* mean fraction of live walkers (weight > 0) over the timed steps */
  double shadow_clip_frac;     /* mean fraction of the live walkers whose exact E_L lies outside the
                                  clip window (running average +- sqrt(2/dt)), over the shadow blocks */
  double one_rdm_weight;       /* cumulativeWeight of the 1-RDM (0 when none was accumulated) */
  int64_t prop_walker_steps;   /* timed steps: sum of the walkers each step propagated       */
  int64_t measured_walkers;    /* timed blocks: sum of the live walkers measured             */
  int64_t exact_walkers;       /* timed surrogate blocks: sum of the exact-set sizes         */
  int64_t restarts;            /* population restarts (restart_every)                         */
  double restart_wall_s;       /* wall seconds of the restarts (not in timed_wall_s)          */
} afq_run_result;

/* ref_up/ref_dn: reference determinant (rhf.txt or uhf.txt by walker type,
 * DQMC/MixedEstimator.cpp:338-351); init_up/init_dn: the right state every
 * walker starts from.  weights_out / energies_out: nsweeps entries each (the
 * samples.dat columns). */
int afq_run_long_prop(const afq_ham* ham, const afq_trial* left, const double* ref_up,
                      const double* ref_dn, const double* init_up, const double* init_dn,
                      const afq_run_params* p, double* weights_out, double* energies_out,
                      afq_run_result* res);

/* Parity hook for the FP64 MFMA tile engine every contraction above uses:
 * C = A B for host row-major A (M x K), B (K x N); C (M x N). */
int afq_debug_gemm_f64(const double* A, const double* B, double* C, int32_t M, int32_t N, int32_t K);

/* Parity hook for the BF16 MFMA tile engine: A, B as above (FP64, split on the
 * device into bf16 hi/lo), C = A B accumulated in FP32 with passes = 3
 * (hi*hi + hi*lo + lo*hi) or 1 (hi*hi). */
int afq_debug_gemm_bf16(const double* A, const double* B, float* C, int32_t M, int32_t N, int32_t K,
                        int32_t passes);

/* Streams `bytes` through a plain copy kernel (k_copy_calib: reads and writes
 * bytes each); a known-size reference for HBM traffic counters. */
int afq_debug_copy(int64_t bytes);

/* Synchronise the context's stream. */
int afq_sync(afq_ctx* ctx);

#ifdef __cplusplus
}
#endif

#endif /* VMC_AFQMC_H */
