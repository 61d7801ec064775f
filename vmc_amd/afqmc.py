"""ctypes binding of the HIP library (vmc_amd/libvmc_afqmc.so, C ABI in
include/vmc_afqmc.h).

There is no CPU fallback: if the library is missing or no device is present the
calls raise.  Build it with `python -m vmc_amd.build` (or __graft_entry__.build()).
"""
import ctypes as C
import os

import numpy as np

from .abi import (AFQ_ENERGY_EXACT, AFQ_PREC_BF16, AFQ_PREC_FP64, AFQ_SURR_MLP, AfqHam, AfqParams, AfqTrial, DP,
                  dptr)

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libvmc_afqmc.so")

_lib = None


class AfqError(RuntimeError):
    pass


def lib():
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise AfqError("HIP library %s not built (run python -m vmc_amd.build)" % LIB_PATH)
        L = C.CDLL(LIB_PATH)
        vp = C.c_void_p
        i32, i64, u64, d = C.c_int32, C.c_int64, C.c_uint64, C.c_double
        L.afq_version.restype = C.c_int
        L.afq_last_error.restype = C.c_char_p
        L.afq_last_error.argtypes = [vp]
        L.afq_create.argtypes = [C.POINTER(AfqHam), C.POINTER(AfqTrial), C.POINTER(AfqParams), C.POINTER(vp)]
        L.afq_destroy.argtypes = [vp]
        L.afq_set_nchol_ene.argtypes = [vp, i32]
        L.afq_set_precision.argtypes = [vp, i32, i32, i32]
        L.afq_prep_prop.argtypes = [vp, DP, DP, DP, DP, d, d]
        L.afq_set_walkers.argtypes = [vp, DP, DP, DP]
        L.afq_get_walkers.argtypes = [vp, DP, DP, DP]
        L.afq_get_weights.argtypes = [vp, DP]
        L.afq_set_weights.argtypes = [vp, DP]
        L.afq_propagate.argtypes = [vp, DP, u64, u64, d, DP, C.POINTER(i64)]
        L.afq_orthogonalize.argtypes = [vp]
        L.afq_measure.argtypes = [vp, i32, d, DP, DP]
        L.afq_ham_and_overlap.argtypes = [vp, DP, i32, i32, DP]
        L.afq_force_bias.argtypes = [vp, DP]
        L.afq_overlap.argtypes = [vp, DP]
        L.afq_comb.argtypes = [vp, d, DP]
        L.afq_rdm_reset.argtypes = [vp]
        L.afq_rdm_accumulate.argtypes = [vp]
        L.afq_get_one_rdm.argtypes = [vp, i32, DP, DP]
        L.afq_stage_times.argtypes = [vp, DP, i32]
        L.afq_sync.argtypes = [vp]
        L.afq_debug_gemm_f64.argtypes = [DP, DP, DP, i32, i32, i32]
        L.afq_debug_copy.argtypes = [i64]
        FP = C.POINTER(C.c_float)
        L.afq_surrogate_init.argtypes = [vp, i32, u64, i64]
        L.afq_surrogate_collect.argtypes = [vp, C.POINTER(i64)]
        L.afq_surrogate_load.argtypes = [vp, C.POINTER(C.c_float), C.POINTER(C.c_float), i64, C.POINTER(i64)]
        L.afq_surrogate_train.argtypes = [vp, i32, i32, d, u64, DP, DP]
        L.afq_surrogate_predict.argtypes = [vp, DP]
        L.afq_surrogate_params.argtypes = [vp, FP, i64, i32]
        L.afq_surrogate_grad.argtypes = [vp, FP, FP, i32, FP, DP]
        L.afq_set_cv.argtypes = [vp, i32, d, d, u64]
        L.afq_set_energy_clip.argtypes = [vp, DP, d]
        L.afq_set_surrogate_kind.argtypes = [vp, i32, i32]
        L.afq_cv_stats.argtypes = [vp, DP]
        L.afq_energy_parts.argtypes = [vp, DP, DP]
        L.afq_surrogate_features.argtypes = [vp, FP]
        L.afq_debug_gemm_bf16.argtypes = [DP, DP, C.POINTER(C.c_float), i32, i32, i32, i32]
        L.afq_set_walkers_uniform.argtypes = [vp, DP, DP, d]
        L.afq_set_clip_centers.argtypes = [vp, DP, i32, d]
        L.afq_block_totals.argtypes = [vp]
        L.afq_debug_cv_force_position.argtypes = [vp, i32]
        _lib = L
    return _lib


STAGES = ["force_bias", "fields", "vhs", "onebody", "green", "weight", "ortho", "exchange", "comb", "taylor",
          "exchange_lp"]


def c2f(a):
    return np.ascontiguousarray(a, dtype=np.complex128).view(np.float64)


def debug_gemm_f64(A, B):
    A = np.ascontiguousarray(A, dtype=np.float64)
    B = np.ascontiguousarray(B, dtype=np.float64)
    M, K = A.shape
    K2, N = B.shape
    assert K == K2
    Cm = np.zeros((M, N))
    rc = lib().afq_debug_gemm_f64(dptr(A), dptr(B), dptr(Cm), M, N, K)
    if rc != 0:
        raise AfqError("debug_gemm: %s" % lib().afq_last_error(None).decode())
    return Cm


def debug_gemm_bf16(A, B, passes=3):
    A = np.ascontiguousarray(A, dtype=np.float64)
    B = np.ascontiguousarray(B, dtype=np.float64)
    M, K = A.shape
    N = B.shape[1]
    Cm = np.zeros((M, N), np.float32)
    rc = lib().afq_debug_gemm_bf16(dptr(A), dptr(B), Cm.ctypes.data_as(C.POINTER(C.c_float)), M, N, K, passes)
    if rc != 0:
        raise AfqError("debug_gemm_bf16: %s" % lib().afq_last_error(None).decode())
    return Cm


def debug_copy(nbytes):
    """Run the plain copy calibration kernel over nbytes (read) + nbytes (write)."""
    if lib().afq_debug_copy(int(nbytes)) != 0:
        raise AfqError("debug_copy: %s" % lib().afq_last_error(None).decode())


class Context:
    """One afq_ctx: a rank's walker population on one GPU."""

    def __init__(self, ham, nwalk, walker_rhf, ref_compat=False, prec_fb=AFQ_PREC_FP64,
                 prec_vhs=AFQ_PREC_FP64, prec_exchange=AFQ_PREC_FP64, device=0, weight_cap=0.0):
        self.h = ham
        self.nwalk = int(nwalk)
        self._hs = ham.ham_struct()
        self._ts = ham.trial_struct()
        self._ps = AfqParams(self.nwalk, int(walker_rhf), int(ref_compat), prec_fb, prec_vhs,
                             prec_exchange, device, weight_cap)
        p = C.c_void_p()
        rc = lib().afq_create(C.byref(self._hs), C.byref(self._ts), C.byref(self._ps), C.byref(p))
        if rc != 0:
            raise AfqError("afq_create(%d): %s" % (rc, lib().afq_last_error(None).decode()))
        self.ptr = p

    @classmethod
    def borrowed(cls, ham, nwalk, walker_rhf, ptr):
        """A view of a context owned elsewhere (a batch's system); never destroyed here."""
        self = cls.__new__(cls)
        self.h = ham
        self.nwalk = int(nwalk)
        self.ptr = ptr
        self._borrowed = True
        return self

    def _chk(self, rc, what):
        if rc != 0:
            raise AfqError("%s(%d): %s" % (what, rc, lib().afq_last_error(self.ptr).decode()))

    def close(self):
        if getattr(self, "_borrowed", False):
            self.ptr = None
            return
        if getattr(self, "ptr", None):
            lib().afq_destroy(self.ptr)
            self.ptr = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def set_precision(self, prec_fb=AFQ_PREC_FP64, prec_vhs=AFQ_PREC_FP64, prec_exchange=AFQ_PREC_FP64):
        self._chk(lib().afq_set_precision(self.ptr, prec_fb, prec_vhs, prec_exchange), "afq_set_precision")

    def set_prop_precision(self, prec_prop=AFQ_PREC_FP64):
        self._chk(lib().afq_set_prop_precision(self.ptr, prec_prop), "afq_set_prop_precision")

    def set_exchange_chunks(self, chunks):
        """Chunks of the Cholesky vectors per (walker, slot) of the pair-wise exchange (0: by shape)."""
        L = lib()
        L.afq_set_exchange_chunks.argtypes = [C.c_void_p, C.c_int32]
        self._chk(L.afq_set_exchange_chunks(self.ptr, int(chunks)), "afq_set_exchange_chunks")

    def set_force_bias_variant(self, v):
        """Split-BF16 force bias: 0 (default) one workgroup per tile and slot with an FP64
        combine, 1 one workgroup per tile over both slots."""
        L = lib()
        L.afq_set_force_bias_variant.argtypes = [C.c_void_p, C.c_int32]
        self._chk(L.afq_set_force_bias_variant(self.ptr, int(v)), "afq_set_force_bias_variant")

    def set_vhs_tile(self, tile):
        """Split-BF16 VHS tile: 0 128 rows single-buffered, 1 256 rows double-buffered,
        2 128 rows double-buffered, 3 (default) and 4 as 0 and 2 with 16-byte output runs
        below the diagonal."""
        L = lib()
        L.afq_set_vhs_tile.argtypes = [C.c_void_p, C.c_int32]
        self._chk(L.afq_set_vhs_tile(self.ptr, int(tile)), "afq_set_vhs_tile")

    def set_exchange3_variant(self, variant):
        """Three-pass split-BF16 exchange: 0 (default) the pair-wise kernel where it applies, 1 the tiled
        kernel, 2 the pair-wise kernel in the VGPR register form."""
        L = lib()
        L.afq_set_exchange3_variant.argtypes = [C.c_void_p, C.c_int32]
        self._chk(L.afq_set_exchange3_variant(self.ptr, int(variant)), "afq_set_exchange3_variant")

    def set_exchange64_variant(self, variant):
        """FP64 exchange kernel: 0 (default) operands straight into registers (from 4 electrons a slot,
        below that as 2 with 8 waves), 1 element loaders, 2 pointer-loader engine with 4 waves."""
        L = lib()
        L.afq_set_exchange64_variant.argtypes = [C.c_void_p, C.c_int32]
        self._chk(L.afq_set_exchange64_variant(self.ptr, int(variant)), "afq_set_exchange64_variant")

    def set_exchange_variant(self, variant):
        """One-pass BF16 exchange kernel: 0 by shape, 1 tiled, 2 pair-wise."""
        self._chk(lib().afq_set_exchange_variant(self.ptr, int(variant)), "afq_set_exchange_variant")

    def set_nchol_ene(self, n):
        self._chk(lib().afq_set_nchol_ene(self.ptr, int(n)), "afq_set_nchol_ene")

    def prep_prop(self, ref_up, ref_dn, dt, ene0=0.0, rdm_up=None, rdm_dn=None):
        ru = np.ascontiguousarray(ref_up, dtype=np.float64)
        rd = np.ascontiguousarray(ref_dn, dtype=np.float64)
        a = None if rdm_up is None else np.ascontiguousarray(rdm_up, dtype=np.float64)
        b = None if rdm_dn is None else np.ascontiguousarray(rdm_dn, dtype=np.float64)
        self._chk(lib().afq_prep_prop(self.ptr, dptr(ru), dptr(rd), dptr(a), dptr(b), dt, ene0),
                  "afq_prep_prop")

    def set_walkers(self, dets, overlaps=None, weights=None):
        d = c2f(dets)
        o = None if overlaps is None else c2f(overlaps)
        w = None if weights is None else np.ascontiguousarray(weights, dtype=np.float64)
        self._chk(lib().afq_set_walkers(self.ptr, dptr(d), dptr(o), dptr(w)), "afq_set_walkers")

    def set_walkers_uniform(self, det, overlap=None, weight=1.0):
        """Every walker a copy of det (one walker in the serial layout), copied on the device."""
        d = c2f(np.asarray(det).reshape(-1))
        o = None if overlap is None else c2f(np.array([overlap]))
        self._chk(lib().afq_set_walkers_uniform(self.ptr, dptr(d), dptr(o), float(weight)),
                  "afq_set_walkers_uniform")

    def set_clip_centers(self, centers=None, halfwidth=0.0):
        c = None if centers is None else np.ascontiguousarray(np.atleast_1d(centers), dtype=np.float64)
        n = 0 if c is None else len(c)
        self._chk(lib().afq_set_clip_centers(self.ptr, dptr(c), n, halfwidth), "afq_set_clip_centers")

    def block_totals(self):
        self._chk(lib().afq_block_totals(self.ptr), "afq_block_totals")

    def step_stats(self):
        st = StepStats()
        L = lib()
        L.afq_get_step_stats.argtypes = [C.c_void_p, C.POINTER(StepStats)]
        self._chk(L.afq_get_step_stats(self.ptr, C.byref(st)), "afq_get_step_stats")
        return {f: getattr(st, f) for f, _ in StepStats._fields_}

    def cv_force_position(self, position):
        """Test hook: every block of the control variate's exact set takes this position
        (position < 0: uniform draws)."""
        self._chk(lib().afq_debug_cv_force_position(self.ptr, int(position)), "afq_debug_cv_force_position")

    def get_walkers(self):
        d = np.zeros((self.nwalk, self.h.mat_size), np.complex128)
        o = np.zeros(self.nwalk, np.complex128)
        w = np.zeros(self.nwalk)
        self._chk(lib().afq_get_walkers(self.ptr, dptr(d.view(np.float64)), dptr(o.view(np.float64)),
                                        dptr(w)), "afq_get_walkers")
        return d, o, w

    def weights(self):
        w = np.zeros(self.nwalk)
        self._chk(lib().afq_get_weights(self.ptr, dptr(w)), "afq_get_weights")
        return w

    def set_weights(self, w):
        w = np.ascontiguousarray(w, dtype=np.float64)
        self._chk(lib().afq_set_weights(self.ptr, dptr(w)), "afq_set_weights")

    def propagate(self, draws=None, eshift=0.0, seed=0, step=0, want_factors=True):
        dr = None if draws is None else np.ascontiguousarray(draws, dtype=np.float64)
        f = np.zeros(self.nwalk) if want_factors else None
        nc = C.c_int64(0)
        self._chk(lib().afq_propagate(self.ptr, dptr(dr), seed, step, eshift, dptr(f), C.byref(nc)),
                  "afq_propagate")
        return f, nc.value

    def orthogonalize(self):
        self._chk(lib().afq_orthogonalize(self.ptr), "afq_orthogonalize")

    def measure(self, delta=0.0, mode=AFQ_ENERGY_EXACT, want_ho=True):
        e = np.zeros(self.nwalk)
        ho = np.zeros((self.nwalk, 2), np.complex128) if want_ho else None
        self._chk(lib().afq_measure(self.ptr, mode, delta, dptr(e),
                                    dptr(None if ho is None else ho.view(np.float64))), "afq_measure")
        return (e, ho) if want_ho else e

    def ham_and_overlap(self, dets, nchol_ene):
        dets = np.atleast_2d(np.asarray(dets, dtype=np.complex128))
        out = np.zeros((dets.shape[0], 2), np.complex128)
        self._chk(lib().afq_ham_and_overlap(self.ptr, dptr(c2f(dets)), dets.shape[0], int(nchol_ene),
                                            dptr(out.view(np.float64))), "afq_ham_and_overlap")
        return out

    def force_bias(self):
        fb = np.zeros((self.nwalk, self.h.nchol), np.complex128)
        self._chk(lib().afq_force_bias(self.ptr, dptr(fb.view(np.float64))), "afq_force_bias")
        return fb

    def overlaps(self):
        o = np.zeros(self.nwalk, np.complex128)
        self._chk(lib().afq_overlap(self.ptr, dptr(o.view(np.float64))), "afq_overlap")
        return o

    def comb(self, zeta):
        t = np.zeros(1)
        self._chk(lib().afq_comb(self.ptr, zeta, dptr(t)), "afq_comb")
        return t[0]

    def rdm_reset(self):
        self._chk(lib().afq_rdm_reset(self.ptr), "afq_rdm_reset")

    def rdm_accumulate(self):
        """One measurement of the mixed-estimator 1-RDM (every walker of nonzero weight)."""
        self._chk(lib().afq_rdm_accumulate(self.ptr), "afq_rdm_accumulate")

    def one_rdm(self, spin_summed):
        """(weighted-average 1-RDM, cumulative weight): N x N if spin_summed, else 2 x N x N."""
        N = self.h.norb
        r = np.zeros((N, N) if spin_summed else (2, N, N))
        cw = np.zeros(1)
        self._chk(lib().afq_get_one_rdm(self.ptr, int(spin_summed), dptr(r), dptr(cw)), "afq_get_one_rdm")
        return r, cw[0]

    def stage_times(self, reset=True):
        ms = np.zeros(len(STAGES))
        self._chk(lib().afq_stage_times(self.ptr, dptr(ms), int(reset)), "afq_stage_times")
        return dict(zip(STAGES, ms))

    def sync(self):
        self._chk(lib().afq_sync(self.ptr), "afq_sync")

    # ---- surrogate control variate
    def surrogate_init(self, hidden=256, seed=1, capacity=0):
        self._chk(lib().afq_surrogate_init(self.ptr, hidden, seed, capacity), "afq_surrogate_init")
        self.hidden = hidden
        self.nfeat = self.h.nchol + 2 * self.h.norb

    def surrogate_collect(self):
        n = C.c_int64(0)
        self._chk(lib().afq_surrogate_collect(self.ptr, C.byref(n)), "afq_surrogate_collect")
        return n.value

    def surrogate_load(self, X, Y):
        X = np.ascontiguousarray(X, np.float32)
        Y = np.ascontiguousarray(Y, np.float32)
        assert X.shape == (len(Y), self.nfeat)
        n = C.c_int64(0)
        fp = C.POINTER(C.c_float)
        self._chk(lib().afq_surrogate_load(self.ptr, X.ctypes.data_as(fp), Y.ctypes.data_as(fp), len(Y),
                                           C.byref(n)), "afq_surrogate_load")
        return n.value

    def surrogate_train(self, epochs=20, batch=512, lr=1e-3, seed=3):
        a, b = C.c_double(0), C.c_double(0)
        self._chk(lib().afq_surrogate_train(self.ptr, epochs, batch, lr, seed, C.byref(a), C.byref(b)),
                  "afq_surrogate_train")
        return a.value, b.value

    def surrogate_predict(self):
        out = np.zeros(self.nwalk)
        self._chk(lib().afq_surrogate_predict(self.ptr, dptr(out)), "afq_surrogate_predict")
        return out

    def _nparams(self):
        F, H = self.nfeat, self.hidden
        dims = [F, H, H, H, 1]
        return dims, sum(dims[l] * dims[l + 1] + dims[l + 1] for l in range(4)) + 2 * F + 2

    def surrogate_params(self, new=None):
        dims, n = self._nparams()
        FP = C.POINTER(C.c_float)
        if new is None:
            buf = np.zeros(n, np.float32)
            self._chk(lib().afq_surrogate_params(self.ptr, buf.ctypes.data_as(FP), n, 0), "afq_surrogate_params")
            return buf
        buf = np.ascontiguousarray(new, dtype=np.float32)
        self._chk(lib().afq_surrogate_params(self.ptr, buf.ctypes.data_as(FP), len(buf), 1), "afq_surrogate_params")

    def surrogate_grad(self, X, t):
        dims, n = self._nparams()
        FP = C.POINTER(C.c_float)
        X = np.ascontiguousarray(X, dtype=np.float32)
        t = np.ascontiguousarray(t, dtype=np.float32)
        ng = n - 2 * dims[0] - 2
        g = np.zeros(ng, np.float32)
        loss = C.c_double(0)
        self._chk(lib().afq_surrogate_grad(self.ptr, X.ctypes.data_as(FP), t.ctypes.data_as(FP), len(t),
                                           g.ctypes.data_as(FP), C.byref(loss)), "afq_surrogate_grad")
        return loss.value, g

    def energy_parts(self):
        e1 = np.zeros(self.nwalk)
        ek = np.zeros(self.nwalk)
        self._chk(lib().afq_energy_parts(self.ptr, dptr(e1), dptr(ek)), "afq_energy_parts")
        return e1, ek

    def features(self):
        F = self.h.nchol + 2 * self.h.norb
        X = np.zeros((self.nwalk, F), np.float32)
        self._chk(lib().afq_surrogate_features(self.ptr, X.ctypes.data_as(C.POINTER(C.c_float))),
                  "afq_surrogate_features")
        return X

    def set_cv(self, subset_inv=16, risk_frac=0.05, fallback_rms=0.0, seed=5):
        self._chk(lib().afq_set_cv(self.ptr, subset_inv, risk_frac, fallback_rms, seed), "afq_set_cv")

    def set_surrogate_kind(self, kind, prec=AFQ_PREC_BF16):
        self._chk(lib().afq_set_surrogate_kind(self.ptr, kind, prec), "afq_set_surrogate_kind")

    def set_energy_clip(self, center=None, halfwidth=0.0):
        c = None if center is None else np.ascontiguousarray(center, dtype=np.float64)
        self._chk(lib().afq_set_energy_clip(self.ptr, dptr(c), halfwidth), "afq_set_energy_clip")

    def cv_stats(self):
        o = np.zeros(6)
        self._chk(lib().afq_cv_stats(self.ptr, dptr(o)), "afq_cv_stats")
        return dict(nsel=o[0], rms=o[1], fallback=o[2], var_sub=o[3], mean_resid=o[4], n_fallback=o[5])


class Batch:
    """Many systems advanced together (afq_batch_*): one context per system, one
    hipGraph launch per step."""

    def __init__(self, hams, walker_rhf, nwalk, device=0):
        L = lib()
        if not hasattr(L, "_batch_bound"):
            vp = C.c_void_p
            L.afq_batch_create.argtypes = [C.c_int32, C.POINTER(AfqHam), C.POINTER(AfqTrial), C.POINTER(AfqParams),
                                           C.POINTER(vp)]
            L.afq_batch_destroy.argtypes = [vp]
            L.afq_batch_context.argtypes = [vp, C.c_int32, C.POINTER(vp)]
            L.afq_batch_capture.argtypes = [vp, C.c_uint64, C.c_int32, C.c_double, C.c_uint64]
            L.afq_batch_step.argtypes = [vp, C.c_int64, DP, DP, DP, C.c_int32, DP]
            L.afq_batch_counts.argtypes = [vp, C.c_void_p, C.c_void_p]
            L.afq_batch_set_lanes.argtypes = [vp, C.c_int32]
            L.afq_batch_launches.argtypes = [vp, C.c_int32, C.POINTER(C.c_int32)]
            L.afq_autotune.argtypes = [vp, C.POINTER(C.c_int32), DP]
            L.afq_set_taylor_variant.argtypes = [vp, C.c_int32]
            L._batch_bound = True
        n = len(hams)
        self.hams = hams
        self.n = n
        hs = (AfqHam * n)(*[h.ham_struct() for h in hams])
        ts = (AfqTrial * n)(*[h.trial_struct() for h in hams])
        ps = (AfqParams * n)(*[AfqParams(nwalk, int(walker_rhf), 0, AFQ_PREC_FP64, AFQ_PREC_FP64, AFQ_PREC_FP64,
                                         device, 0.0) for _ in hams])
        self.ptr = C.c_void_p()
        rc = L.afq_batch_create(n, hs, ts, ps, C.byref(self.ptr))
        if rc:
            raise AfqError("afq_batch_create(%d): %s" % (rc, L.afq_last_error(None).decode()))
        self.ctx = []
        for i, h in enumerate(hams):
            cp = C.c_void_p()
            L.afq_batch_context(self.ptr, i, C.byref(cp))
            self.ctx.append(Context.borrowed(h, nwalk, walker_rhf, cp))

    def autotune(self):
        out = []
        for c in self.ctx:
            ch = C.c_int32(0)
            ms = np.zeros(3)
            c._chk(lib().afq_autotune(c.ptr, C.byref(ch), dptr(ms)), "afq_autotune")
            out.append((ch.value, ms))
        return out

    def set_lanes(self, lanes):
        """Grouped launches on `lanes` streams (default 1); 0: one graph branch per system."""
        rc = lib().afq_batch_set_lanes(self.ptr, int(lanes))
        if rc:
            raise AfqError("afq_batch_set_lanes(%d): %s" % (rc, lib().afq_last_error(None).decode()))

    def launches(self, qr=False):
        """Kernel launches in one captured step (-1 for the one-branch-per-system form)."""
        v = C.c_int32()
        rc = lib().afq_batch_launches(self.ptr, int(qr), C.byref(v))
        if rc:
            raise AfqError("afq_batch_launches(%d): %s" % (rc, lib().afq_last_error(None).decode()))
        return v.value

    def capture(self, seed, ortho_steps, clip_halfwidth, first_step=1):
        rc = lib().afq_batch_capture(self.ptr, seed, ortho_steps, clip_halfwidth, first_step)
        if rc:
            raise AfqError("afq_batch_capture(%d): %s" % (rc, lib().afq_last_error(None).decode()))

    def step(self, step, eshift, zeta, center, graph=True):
        tot = np.zeros(2 * self.n)
        args = [np.ascontiguousarray(x, dtype=np.float64) for x in (eshift, zeta, center)]
        rc = lib().afq_batch_step(self.ptr, step, dptr(args[0]), dptr(args[1]), dptr(args[2]), int(graph),
                                  dptr(tot))
        if rc:
            raise AfqError("afq_batch_step(%d): %s" % (rc, lib().afq_last_error(None).decode()))
        return tot.reshape(self.n, 2)

    def counts(self):
        """(walkers propagated, walkers live) per system in the last step."""
        prop, live = np.zeros(self.n, dtype=np.int64), np.zeros(self.n, dtype=np.int64)
        rc = lib().afq_batch_counts(self.ptr, prop.ctypes.data, live.ctypes.data)
        if rc:
            raise AfqError("afq_batch_counts(%d): %s" % (rc, lib().afq_last_error(None).decode()))
        return prop, live

    def close(self):
        if self.ptr:
            lib().afq_batch_destroy(self.ptr)
            self.ptr = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


AFQ_RNG_REPLAY = 0
AFQ_RNG_DEVICE = 1


class RunParams(C.Structure):
    _fields_ = [
        ("seed", C.c_int64), ("dt", C.c_double), ("nsteps", C.c_int32), ("nsweeps", C.c_int32),
        ("ortho_steps", C.c_int32), ("burn_iter", C.c_int32), ("nwalk", C.c_int32),
        ("nranks", C.c_int32), ("walker_rhf", C.c_int32), ("ref_compat", C.c_int32),
        ("cholesky_threshold", C.c_double), ("ene0_guess", C.c_double), ("weight_cap", C.c_double),
        ("max_steps", C.c_int32), ("rng_mode", C.c_int32), ("warmup_steps", C.c_int32),
        ("prec_fb", C.c_int32), ("prec_vhs", C.c_int32), ("prec_exchange", C.c_int32),
        ("energy_mode", C.c_int32), ("device", C.c_int32),
        ("surrogate_train_steps", C.c_int32), ("surrogate_hidden", C.c_int32),
        ("surrogate_epochs", C.c_int32), ("subset_inv", C.c_int32), ("fallback_rms", C.c_double),
        ("risk_frac", C.c_double), ("shadow_exact", C.c_int32), ("surrogate_kind", C.c_int32),
        ("surrogate_prec", C.c_int32), ("prec_prop", C.c_int32), ("one_rdm_out", DP),
        ("rdm_background", DP), ("restart_every", C.c_int32),
    ]


class RunResult(C.Structure):
    _fields_ = [("ref_energy", C.c_double), ("nchol_ene", C.c_int32), ("delta", C.c_double),
                ("n_large_deviations", C.c_int64), ("prop_time", C.c_double),
                ("ene_time", C.c_double), ("timed_steps", C.c_int64), ("timed_wall_s", C.c_double),
                ("stage_ms", C.c_double * len(STAGES)), ("train_rmse", C.c_double), ("valid_rmse", C.c_double),
                ("cv_var_sub", C.c_double), ("cv_rms", C.c_double), ("cv_fallbacks", C.c_int64),
                ("train_samples", C.c_int64), ("est_var", C.c_double), ("shadow_n", C.c_int64),
                ("shadow_shift", C.c_double), ("shadow_var", C.c_double), ("shadow_est_var", C.c_double),
                ("shadow_wall_s", C.c_double), ("live_frac", C.c_double), ("shadow_clip_frac", C.c_double),
                ("one_rdm_weight", C.c_double), ("prop_walker_steps", C.c_int64), ("measured_walkers", C.c_int64),
                ("exact_walkers", C.c_int64), ("restarts", C.c_int64), ("restart_wall_s", C.c_double)]


class StepStats(C.Structure):
    """afq_step_stats: the population statistics kept on the device."""
    _fields_ = [("total_weight", C.c_double), ("n_propagated", C.c_int64), ("n_live", C.c_int64),
                ("n_capped", C.c_int64), ("block_weight", C.c_double), ("block_wsum", C.c_double),
                ("block_var", C.c_double), ("n_measured", C.c_int64), ("n_clipped", C.c_int64),
                ("n_nonfinite", C.c_int64), ("n_exact", C.c_int64), ("cv_rms", C.c_double),
                ("cv_var_sub", C.c_double), ("cv_mean_resid", C.c_double), ("cv_fallback", C.c_int32),
                ("comb_total", C.c_double)]


def run_long_prop(ham, ref_up, ref_dn, init_up, init_dn, *, seed, dt, nsteps, nsweeps, ortho_steps,
                  nwalk, nranks=1, walker_rhf, ref_compat=False, cholesky_threshold=1e-3,
                  burn_iter=0, ene0_guess=1e10, weight_cap=0.0, max_steps=0,
                  rng_mode=AFQ_RNG_REPLAY, warmup_steps=0, prec_fb=AFQ_PREC_FP64,
                  prec_vhs=AFQ_PREC_FP64, prec_exchange=AFQ_PREC_FP64,
                  energy_mode=AFQ_ENERGY_EXACT, device=0, surrogate_train_steps=0, surrogate_hidden=256,
                  surrogate_epochs=20, subset_inv=16, fallback_rms=0.0, risk_frac=0.05, shadow_exact=False,
                  surrogate_kind=AFQ_SURR_MLP, surrogate_prec=AFQ_PREC_BF16, prec_prop=AFQ_PREC_FP64,
                  one_rdm=None, background_rdm=None, restart_every=0):
    """calcMixedEstimatorLongProp on the GPU; returns (weights, energies, RunResult).
    one_rdm: None, or a float64 array that receives the mixed-estimator 1-RDM
    (N x N for an RHF trial, 2 x N x N for a UHF trial).  background_rdm: None, or
    the 2 x N x N (up, down) density of spinRDM.0.0.txt for the mean-field shifts."""
    L = lib()
    if not hasattr(L, "_run_bound"):
        L.afq_run_long_prop.argtypes = [C.POINTER(AfqHam), C.POINTER(AfqTrial), DP, DP, DP, DP,
                                        C.POINTER(RunParams), DP, DP, C.POINTER(RunResult)]
        L._run_bound = True
    hs, ts = ham.ham_struct(), ham.trial_struct()
    p = RunParams(seed, dt, nsteps, nsweeps, ortho_steps, burn_iter, nwalk, nranks, int(walker_rhf),
                  int(ref_compat), cholesky_threshold, ene0_guess, weight_cap, max_steps, rng_mode,
                  warmup_steps, prec_fb, prec_vhs, prec_exchange, energy_mode, device,
                  surrogate_train_steps, surrogate_hidden, surrogate_epochs, subset_inv, fallback_rms,
                  risk_frac, int(shadow_exact), surrogate_kind, surrogate_prec, prec_prop, dptr(one_rdm),
                  dptr(None if background_rdm is None else np.ascontiguousarray(background_rdm, dtype=np.float64)),
                  int(restart_every))
    w = np.zeros(nsweeps)
    e = np.zeros(nsweeps)
    res = RunResult()
    arrs = [np.ascontiguousarray(a, dtype=np.float64) for a in (ref_up, ref_dn, init_up, init_dn)]
    rc = L.afq_run_long_prop(C.byref(hs), C.byref(ts), *[dptr(a) for a in arrs], C.byref(p),
                             dptr(w), dptr(e), C.byref(res))
    if rc != 0:
        raise AfqError("afq_run_long_prop(%d): %s" % (rc, L.afq_last_error(None).decode()))
    return w, e, res
