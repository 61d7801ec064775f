#!/usr/bin/env python3
"""Throughput of the phaseless-AFQMC walker step on one MI355X.

A step is one pass of the walker step over the whole population: force bias,
field draws (device counter-based RNG), VHS, Taylor propagation, Green's
function / overlap, phaseless weights, population control, QR every 5 steps,
and the local energy of every walker.  Inputs are resident in HBM before the
timed region.  Paths:

  fp64               exact FP64 local energy of every walker;
  mixed_exchange_cv  force bias, VHS and Taylor products in split BF16 (three
                     passes, FP32 accumulation); control variate: the exchange in one BF16 MFMA
                     pass on every live walker, exact FP64 on a random 1/subset_inv
                     of them (Horvitz-Thompson correction, unbiased); the headline;
  mlp_cv             control variate with the learned MLP surrogate, trained on
                     the GPU from the first exact steps.

Both control-variate paths also measure every block exactly in FP64 outside the
timings ("shadow"), which gives the energy shift on identical walkers.

Workload (default): N=300 orbitals, 60+60 electrons, 1200 Cholesky vectors,
UHF trial, 4096 walkers, dt=0.005 -- synthetic Hamiltonian (vmc_amd.synthetic).

Prints one JSON line.  `python bench.py --gpus N` with N > 1 exits: this build
runs on a single GPU.
"""
import argparse
import collections
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import numpy as np  # noqa: E402

METRIC = ("walker-steps/s/GPU mixed-prec+surrogate vs plain FP64, at ≤0.1 mHa energy shift")
PEAK_FP64_TFLOPS = 78.6


def exchange_flops(spec, nwalk):
    """Algorithmic FLOPs of one exchange launch: per walker and spin
    4 G n^2 N (f = R_g theta) + 8 G n^2 (sum_ij f_ij f_ji)."""
    N, G = spec["norb"], spec["nchol"]
    nsp = [spec["nalpha"]] if spec["walker_rhf"] else [spec["nalpha"], spec["nbeta"]]
    return nwalk * sum(4.0 * G * n * n * N + 8.0 * G * n * n for n in nsp)


def flops_per_walker_step(spec, ortho=5, energy=True):
    """Algorithmic real FLOPs of one walker-step (complex x real MAC = 4, complex x
    complex MAC = 8), E_L evaluated every step."""
    N, G = spec["norb"], spec["nchol"]
    T = N * (N + 1) / 2
    nsp = [spec["nalpha"]] if spec["walker_rhf"] else [spec["nalpha"], spec["nbeta"]]
    f = 0.0
    for n in nsp:
        f += 4 * n * n * N + 16 * n ** 3 + 8 * N * n * n      # overlap matrix, inverse, theta
        f += 4 * n * N * G                                     # force bias
        f += 48 * N * N * n                                    # 2 one-body + 5 Taylor products
        f += 4 * n * n * N + 6 * n ** 3                        # new overlap
        f += 16 * (2 * N * n * n - 2.0 / 3.0 * n ** 3) / ortho  # QR, amortised
    f += 4 * T * G                                             # VHS
    if energy:
        for n in nsp:
            f += 4 * G * n * n * N + 8 * G * n * n + 2 * G * n
            f += 4 * n * n * N + 16 * n ** 3 + 8 * N * n * n + 4 * N * n
    return f


def split_flops(spec, ortho=5):
    """Algorithmic FLOPs of one walker-step by part and by the precision the split-BF16
    path runs them in: {(part, prec): flops} with part "prop" (every walker
    propagated) or "meas" (every walker measured) and prec "bf16x3" (force bias, VHS,
    one-body and Taylor products, exchange) or "fp64" (the rest)."""
    N, G = spec["norb"], spec["nchol"]
    T = N * (N + 1) / 2
    nsp = [spec["nalpha"]] if spec["walker_rhf"] else [spec["nalpha"], spec["nbeta"]]
    prop = flops_per_walker_step(spec, ortho, energy=False)
    meas = flops_per_walker_step(spec, ortho) - prop
    prop_lp = 4 * T * G + sum(4 * n * N * G + 48 * N * N * n for n in nsp)
    meas_lp = sum(4 * G * n * n * N + 8 * G * n * n for n in nsp)
    return {("prop", "bf16x3"): prop_lp, ("prop", "fp64"): prop - prop_lp,
            ("meas", "bf16x3"): meas_lp, ("meas", "fp64"): meas - meas_lp}


from vmc_amd.afqmc import STAGES  # noqa: E402
PEAKS = {"fp64": 78.6, "bf16": 2500.0, "fp8": 5000.0}
PREC_NAMES = {0: "fp64", 2: "bf16x3", 3: "bf16", 4: "fp8"}


RESTART_EVERY = 5


def run_path(ham, spec, total_steps, warmup, **kw):
    """Driver run with E_L every step (nsteps=1), device RNG; the first `warmup`
    steps are excluded from timing.  Every RESTART_EVERY steps the population restarts
    at the trial determinant (outside the timings), so every timed step propagates a
    live population: left alone, these strongly coupled systems lose weight every step
    until the comb leaves every walker below the propagation threshold (1e-8) for good.
    Throughput counts the walkers actually propagated (weight > 1e-8 at the step's
    start), as the driver reports them."""
    from vmc_amd.afqmc import AFQ_RNG_DEVICE, run_long_prop
    W = spec["nwalk"]
    w, e, res = run_long_prop(
        ham, ham.phi_up, ham.phi_dn, ham.phi_up, ham.phi_dn, seed=20261202, dt=spec["dt"], nsteps=1,
        nsweeps=total_steps + 1, ortho_steps=spec["ortho"], nwalk=W, nranks=1,
        walker_rhf=spec["walker_rhf"], cholesky_threshold=0.0, rng_mode=AFQ_RNG_DEVICE,
        warmup_steps=warmup, restart_every=RESTART_EVERY, **kw)
    k = int(res.timed_steps)
    wall = float(res.timed_wall_s)
    ms = 1e3 * wall / k
    n_prop = int(res.prop_walker_steps)
    return dict(walker_steps_per_s=n_prop / wall, ms_per_step=ms, steps=k, energies=np.array(e),
                propagated_per_step=n_prop / k, measured_per_step=int(res.measured_walkers) / k,
                exact_per_step=int(res.exact_walkers) / k, restarts=int(res.restarts),
                restart_wall_s=float(res.restart_wall_s),
                weights=np.array(w), stage_ms_per_step={n: v / k for n, v in zip(STAGES, res.stage_ms)},
                est_var=float(res.est_var), err_per_sqrt_s=float(np.sqrt(res.est_var * ms * 1e-3)),
                train_rmse=float(res.train_rmse), valid_rmse=float(res.valid_rmse),
                cv_var_sub=float(res.cv_var_sub), cv_rms=float(res.cv_rms),
                cv_fallbacks=int(res.cv_fallbacks), train_samples=int(res.train_samples),
                shadow_n=int(res.shadow_n), shadow_shift=float(res.shadow_shift),
                shadow_var=float(res.shadow_var), shadow_est_var=float(res.shadow_est_var),
                shadow_wall_s=float(res.shadow_wall_s), live_frac=float(res.live_frac),
                shadow_clip_frac=float(res.shadow_clip_frac))


HBM_PEAK_GBS = 8000.0


def fused_prop(spec):
    """Whether the split propagation runs as the fused k_prop_split (N <= 384)."""
    return -(-spec["norb"] // 16) <= 8 * 3


def fused_prop_shape(spec):
    """(row tiles per wave, column tiles per block) of k_prop_split, as the library picks them."""
    ncol = spec["nalpha"] + (0 if spec["walker_rhf"] else spec["nbeta"])
    rt = -(-spec["norb"] // 16)
    mt = -(-rt // 8)
    ctot = -(-ncol // 8)
    nblk = -(-ctot // 4)
    return mt, -(-ctot // nblk)


def stage_rooflines(spec, path, n_exact):
    """Roofline of each stage of one step (per launch for the kernels that launch
    several times).  Algorithmic FLOPs and HBM bytes per launch give two lower
    bounds on the time, FLOPs x passes / MFMA peak and bytes / 8 TB/s; the larger
    one names the bound, and `achieved` is the algorithmic rate in that unit.
    The work of a stage counts only the walkers it processed, per step on average:
    the propagation (VHS, one-body, Taylor, overlap and inverse) the walkers
    propagated, theta and the force bias the walkers still alive after the weight
    update, the reduced-precision exchange the walkers measured and the FP64 exchange
    n_exact of them."""
    N, G = spec["norb"], spec["nchol"]
    T = N * (N + 1) / 2
    nsp = [spec["nalpha"]] if spec["walker_rhf"] else [spec["nalpha"], spec["nbeta"]]
    ncol = sum(nsp)
    ms = N * ncol                      # complex elements of a walker's orbitals
    Wp = path["propagated_per_step"]                  # walkers propagated per step
    Wl = spec["nwalk"] * path.get("live_frac", 1.0)   # alive after the weight update
    Np = (N + 7) // 8 * 8
    st = path["stage_ms_per_step"]
    out = {}

    def add(name, kernel, flops, nbytes, launches, prec, symbol=None, passes=1, **extra):
        ms_l = st.get(name, 0.0) / launches
        if ms_l <= 0:
            return
        f, b = flops / launches, nbytes / launches
        t_mfma = f * passes / (PEAKS[prec] * 1e12)
        t_hbm = b / (HBM_PEAK_GBS * 1e9)
        if t_hbm > t_mfma:
            ach = b / (ms_l * 1e-3) / 1e9
            r = dict(bound="hbm", achieved=ach, peak=HBM_PEAK_GBS, unit="GB/s", frac=ach / HBM_PEAK_GBS)
        else:
            ach = f / (ms_l * 1e-3) / 1e12
            r = dict(bound="mfma", achieved=ach, peak=PEAKS[prec], unit="TFLOP/s", frac=ach / PEAKS[prec])
        r.update(kernel=kernel, symbol=symbol, launch_ms=ms_l, flops_per_launch=f, bytes_per_launch=b,
                 precision=prec, passes=passes, flops_per_step=flops, **extra)
        out[name] = r

    # exchange: the rotated Cholesky once per launch + theta of each walker measured
    if path["exchange_prec"] == "fp64":
        extra = {}
        if path.get("surrogate_prec"):
            # the exact subset of the control variate; the HBM counter summary keeps its
            # dispatches apart from the unclipped shadow measurements on the same kernel
            extra["profile_row"] = "k_exchange (exact subset)"
        add("exchange", "k_exchange64 (FP64 MFMA)", exchange_flops(spec, n_exact),
            8.0 * G * ms + 16.0 * ms * n_exact, 1, "fp64", symbol="k_exchange64", walkers=n_exact, **extra)
    else:
        nmax3 = max(nsp)
        if 12 < nmax3 <= 64 and (Np + 31) // 32 * 32 <= 448:
            kname3 = "k_exchange_pw2 (3-pass split BF16 MFMA, pair-wise, exact level)"
            sym3 = "void k_exchange_pw2x3<%d, 2, 2>" % (-(-nmax3 // 16))
        else:
            kname3, sym3 = "k_exchange_bf16 (3-pass split BF16 MFMA)", "void k_exchange_bf16<2>"
        add("exchange", kname3, exchange_flops(spec, n_exact),
            4.0 * G * ncol * Np + 8.0 * ncol * Np * n_exact, 1, "bf16", symbol=sym3,
            passes=3, walkers=n_exact)
    if path.get("surrogate_prec") == "fp8":
        nl = path["measured_per_step"]
        Npq = (N + 15) // 16 * 16
        add("exchange_lp", "k_exchange_q8 (e4m3 MFMA, per-Cholesky-vector scale, surrogate level)",
            exchange_flops(spec, nl), G * ncol * Npq + 2 * ncol * Npq * nl, 1, "fp8", symbol="k_exchange_q8",
            walkers=nl)
    elif path.get("surrogate_prec"):
        passes = 3 if path["surrogate_prec"] == "bf16x3" else 1
        nl = path["measured_per_step"]
        nmax = max(nsp)
        if passes == 1 and nmax <= 64 and (Np + 31) // 32 * 32 <= 448:
            # the pair-wise kernel, two waves per SIMD: theta of a walker in LDS, R in
            # fragment order, f_ij f_ji in registers
            kname = "k_exchange_pw2 (1-pass BF16 MFMA, R in fragment order, pair sums in registers, surrogate level)"
            sym = "void k_exchange_pw2<%d, 8, false>" % (-(-nmax // 16))
        elif passes == 1 and nmax <= 64 and (Np + 31) // 32 * 32 <= 512:
            # the pair-wise kernel: theta of a walker in LDS, f_ij f_ji in registers
            kname = "k_exchange_pw (1-pass BF16 MFMA, pair sums in registers, surrogate level)"
            sym = "void k_exchange_pw<%d>" % (-(-nmax // 16))
        else:
            kname = "k_exchange_bf16 (%d-pass BF16 MFMA, surrogate level)" % passes
            sym = "void k_exchange_bf16<%d>" % (2 if passes == 3 else 1)
        add("exchange_lp", kname, exchange_flops(spec, nl),
            2.0 * (2 if passes == 3 else 1) * (G * ncol * Np + 2 * ncol * Np * nl),
            1, "bf16", symbol=sym, passes=passes, walkers=nl)
    # Taylor: V (both planes) once, t in, t out, the accumulator read and written, per walker and product
    tay_bytes = Wp * (16.0 * N * N + 4 * 16.0 * ms) * 5
    if path.get("fb_vhs_prec", "fp64") == "fp64":
        wide = ncol > 64
        if st.get("onebody", 0.0) <= 0.0:
            # both one-body factors and the five products in one kernel: V once per product, the orbitals once
            add("taylor", "k_prop64 (E (sum_k V^k/k!) E psi, fused, FP64 MFMA)", Wp * (40.0 + 8.0) * N * N * ncol,
                Wp * (5 * 16.0 * N * N + 32.0 * ms), 1, "fp64", symbol="k_prop64")
        else:
            add("taylor", "k_taylor (5 complex V t products, FP64 MFMA)", Wp * 40.0 * N * N * ncol, tay_bytes, 5,
                "fp64", symbol=("void k_taylor<%s>" % ("true" if N % 2 == 0 else "false")) if wide
                else "void k_vmul<64, 128, 2, 2>")
        add("force_bias", "k_fb64 (FP64 MFMA)", Wl * 4.0 * ncol * N * G, 8.0 * G * ms + Wl * 16.0 * (ms + G),
            1, "fp64", symbol="k_fb64")
        add("vhs", "k_vhs64 (FP64 MFMA)", Wp * 4.0 * T * G, 8.0 * G * T + Wp * 16.0 * (G + N * N), 1, "fp64",
            symbol="k_vhs64")
    else:
        Nq = (N + 15) // 16 * 16
        vb, ub = 8.0 * Nq * N, 8.0 * ncol * Nq
        if fused_prop(spec):
            # k_prop_split: both one-body factors and the 5 Horner steps in one kernel; the
            # walker's orbitals are read and written once (FP64), V (hi, lo: 8 Nq N bytes)
            # once per Horner step, D is shared by all walkers
            mt, ct = fused_prop_shape(spec)
            add("taylor", "k_prop_split (E (sum_k V^k/k!) E psi, fused, 3-pass split BF16 MFMA)",
                Wp * (40.0 + 8.0) * N * N * ncol, Wp * (5 * vb + 32.0 * ms), 1, "bf16",
                symbol="void k_prop_split<%d, %d>" % (mt, ct), passes=3)
        else:
            # Horner steps on split operands: V, u in, t0 and u out (4 planes of bf16:
            # 8 ncol Nq bytes each); the last step adds the FP64 t0 and writes FP64
            tay_split = Wp * (4 * (vb + 3 * ub) + (vb + ub + 32.0 * ms))
            add("taylor", "k_taylor_h (5 Horner steps u = t0 + V u / p, 3-pass split BF16 MFMA)",
                Wp * 40.0 * N * N * ncol, tay_split, 5, "bf16", symbol="void k_taylor_h<%d, %d>" % (
                    5 if -(-N // 160) * 160 < -(-N // 128) * 128 else 4, 1 if ncol <= 32 else 2 if ncol <= 64 else 4),
                passes=3)
        add("force_bias", "k_theta_split + k_force_bias_bf16<2> (3-pass split BF16 MFMA)", Wl * 4.0 * ncol * N * G,
            4.0 * G * ncol * Np + Wl * (16.0 * ms + 8.0 * ncol * Np + 16.0 * G), 1, "bf16",
            symbol="void k_force_bias_bf16<2>", passes=3)
        add("vhs", "k_fields_split + k_vhs_bf16<2> (3-pass split BF16 MFMA)", Wp * 4.0 * T * G,
            4.0 * G * T + Wp * (24.0 * G + 8.0 * ((N + 15) // 16 * 16) * N), 1, "bf16",
            symbol="void k_vhs_bf16<2, 3>", passes=3)
    if path.get("fb_vhs_prec", "fp64") != "fp64" and fused_prop(spec):
        pass   # the one-body factors run inside k_prop_split (the taylor stage)
    elif path.get("fb_vhs_prec", "fp64") == "fp64":
        add("onebody", "k_expmul (E psi, FP64 MFMA)", Wp * 8.0 * N * N * ncol, Wp * 3 * 16.0 * ms, 2 * len(nsp),
            "fp64", symbol="k_expmul")
    else:
        # E x = x + (E - I) x: x read (FP64), E x written (FP64; before the series also split)
        mi = 5 if -(-N // 160) * 160 < -(-N // 128) * 128 else 4
        add("onebody", "k_onebody_split (E x = x + D x, D x in 3-pass split BF16 MFMA)", Wp * 8.0 * N * N * ncol,
            Wp * (40.0 + 32.0) * ms, 2 * len(nsp), "bf16", symbol="void k_onebody_split<%d>" % mi, passes=3)
    # S = Phi^T psi and its inverse for the walkers propagated, theta = psi S^-1 for the
    # walkers still alive
    add("green", "k_overlap + k_invert + k_theta (FP64 MFMA + Gauss-Jordan)",
        sum(Wp * (4 * n * n * N + 16 * n ** 3) + Wl * 8 * N * n * n for n in nsp), (Wp + Wl) * 16.0 * ms, 1,
        "fp64", symbol="k_theta")
    return out


PROFILE_HBM = os.path.join(ROOT, "profiles", "walker_step_N300_G1200_W4096_hbm_counters.md")


def profiled_traffic(workload, kernel):
    """HBM bytes per launch (calibrated FETCH_SIZE + WRITE_SIZE) of a kernel from the
    committed rocprofv3 counter summary of this workload, or None."""
    if workload != "c4" or not os.path.exists(PROFILE_HBM):
        return None
    for line in open(PROFILE_HBM):
        cells = [c.strip() for c in line.strip().strip("|").split("|")]
        if len(cells) == 7 and cells[0] == kernel:
            try:
                return float(cells[6]) * 2 ** 20   # fetch + write over the timed steps' dispatches
            except ValueError:
                return None
    return None


def cv_summary(mx, fp64):
    """Energy shift and statistical efficiency of a control-variate path.

    On identical walkers (a shadow FP64 measurement of every surrogate block,
    outside the timings): shift = mean(E_cv - E_fp64) per block with its standard
    error (the control-variate noise is independent from block to block).  The
    error per sqrt(wall-second) ratio charges that noise on top of the FP64
    estimator's own per-block variance with no credit for autocorrelation of the
    latter, so it is an upper bound."""
    n = mx["shadow_n"]
    sem = float(np.sqrt(mx["shadow_var"] / n)) if n > 1 else None
    ratio = None
    if mx["shadow_est_var"] > 0:
        ratio = float(np.sqrt((1.0 + mx["shadow_var"] / mx["shadow_est_var"])
                              * mx["ms_per_step"] / fp64["ms_per_step"]))
    return dict(energy_shift_mha=1e3 * mx["shadow_shift"],
                energy_shift_sem_mha=None if sem is None else 1e3 * sem,
                energy_shift_blocks=n,
                cv_noise_per_block_mha=1e3 * float(np.sqrt(mx["shadow_var"])),
                clipped_fraction=mx.get("shadow_clip_frac"),
                fp64_error_per_block_mha=1e3 * float(np.sqrt(mx["shadow_est_var"])),
                speedup_vs_fp64=mx["walker_steps_per_s"] / fp64["walker_steps_per_s"],
                err_per_sqrt_s_ratio=ratio)


def host_cores():
    """Host cores this process may use, capped at 16: the one-GPU share of the host that
    the GPU box gives a job (its OMP_NUM_THREADS), whatever the node's nproc."""
    try:
        n = len(os.sched_getaffinity(0))
    except AttributeError:
        n = os.cpu_count() or 1
    return max(1, min(16, n, int(os.environ.get("OMP_NUM_THREADS", "16") or 16)))


def precision_weighted_peak(rooflines):
    """sum F_i / sum (F_i passes_i / P_i) over the stages (TFLOP/s): the rate a step whose
    stages all ran at their precision's MFMA peak would reach on algorithmic FLOPs."""
    num = sum(r["flops_per_step"] for r in rooflines.values())
    den = sum(r["flops_per_step"] * r["passes"] / PEAKS[r["precision"]] for r in rooflines.values())
    return num / den if den > 0 else 0.0


def deterministic_shift(ham, spec, subset_inv, exact_prec, nsteps=4):
    """Energy shift of the headline path without sampling noise, on the workload's own
    system and population size, outside the timings:

    * control variate: averaged over the subset_inv within-block positions of its exact
      set, the estimate is every walker's energy at the exact level (the Horvitz-Thompson
      identity); the residual of that block energy against the FP64 one, with the clip of
      the population control, is its shift: zero up to round-off with the FP64 exact level,
      the exact level's own error with the split-BF16 one (exact_prec);
    * propagation: the same walkers and the same device fields propagated nsteps steps in
      FP64 and in split BF16, both measured in FP64; the weighted block energies differ by
      the shift the reduced-precision propagation makes (per step, mHa).
    Each is reported with the clip and without it: where most energies reach the clip the
    clipped figures are small by construction, and the unclipped ones carry the check."""
    from vmc_amd.abi import AFQ_ENERGY_SURROGATE, AFQ_PREC_BF16, AFQ_PREC_BF16X3, AFQ_PREC_FP64, AFQ_SURR_EXCHANGE
    from vmc_amd.afqmc import Context
    W, dt = spec["nwalk"], spec["dt"]
    det = ham.serial_det(ham.phi_up, ham.phi_dn)
    half = np.sqrt(2.0 / dt)
    ctx = [Context(ham, W, spec["walker_rhf"]) for _ in range(2)]
    try:
        for k, c in enumerate(ctx):
            c.prep_prop(ham.phi_up, ham.phi_dn, dt)
            c.set_walkers_uniform(det)
            if k == 1:
                c.set_precision(prec_fb=AFQ_PREC_BF16X3, prec_vhs=AFQ_PREC_BF16X3)
                c.set_prop_precision(AFQ_PREC_BF16X3)
        e0 = ctx[0].measure(want_ho=False)
        eshift = float(np.mean(e0))
        shifts, shifts_raw = [], []
        for step in range(1, nsteps + 1):
            for c in ctx:
                c.propagate(None, eshift, seed=7, step=step, want_factors=False)
            e = [c.measure(want_ho=False) for c in ctx]
            w = [c.weights() for c in ctx]
            eb = [np.sum(wi * np.clip(ei, eshift - half, eshift + half)) / np.sum(wi) for wi, ei in zip(w, e)]
            shifts.append(1e3 * (eb[1] - eb[0]))
            eb = [np.sum(wi * ei) / np.sum(wi) for wi, ei in zip(w, e)]
            shifts_raw.append(1e3 * (eb[1] - eb[0]))
        # the control variate on the FP64 context's population after those steps, combed so
        # that every walker is live and the blocks of the exact set are all full
        c = ctx[0]
        c.comb(0.5)
        e_exact = c.measure(want_ho=False)
        w = c.weights()
        live = w != 0
        center = float(np.median(e_exact[live]))
        ref = np.where(live, np.clip(e_exact, center - half, center + half), 0.0)
        level = {}
        if exact_prec != AFQ_PREC_FP64:
            # the exact level's own shift: every walker's energy with that exchange
            c.set_precision(prec_exchange=exact_prec)
            e_lvl = c.measure(want_ho=False)
            ref_lvl = np.where(live, np.clip(e_lvl, center - half, center + half), 0.0)
            level = dict(exact_level_shift_mha=float(1e3 * np.sum(w * (ref_lvl - ref)) / np.sum(w)),
                         exact_level_unclipped_shift_mha=float(1e3 * np.sum(w * (e_lvl - e_exact)) / np.sum(w)),
                         exact_level_max_walker_diff_ha=float(np.max(np.abs(e_lvl - e_exact)[live])))
        c.set_surrogate_kind(AFQ_SURR_EXCHANGE, AFQ_PREC_BF16)

        def cv_average():
            acc = np.zeros(W)
            for pos in range(subset_inv):
                c.set_cv(subset_inv=subset_inv, risk_frac=0.0, seed=3)
                c.cv_force_position(pos)
                acc += c.measure(mode=AFQ_ENERGY_SURROGATE, want_ho=False)
            return acc / subset_inv

        c.set_clip_centers([center], half)
        avg = cv_average()
        # the same without the clip: on a workload whose energies mostly reach the clip the
        # clipped residual is small by construction, the raw one is not
        c.set_clip_centers(None)
        avg_raw = cv_average()
        nl = int(live.sum())
        exact_avg = nl % subset_inv == 0
        res = 1e3 * (np.sum(w * avg) - np.sum(w * ref)) / np.sum(w)
        res_raw = 1e3 * np.sum(w * np.where(live, avg_raw - e_exact, 0.0)) / np.sum(w)
        clipped = float(np.mean(np.abs(e_exact[live] - center) > half)) if nl else 0.0
        return dict(cv_expectation_residual_mha=float(res), cv_expectation_unclipped_residual_mha=float(res_raw),
                    exact_level=PREC_NAMES[exact_prec], **level,
                    clipped_fraction=clipped,
                    cv_expectation_max_walker_residual_ha=float(np.max(np.abs(avg - ref)[live])) if nl else 0.0,
                    cv_expectation_exact_average=bool(exact_avg), live_walkers=nl,
                    propagation_shift_mha=[float(x) for x in shifts],
                    propagation_unclipped_shift_mha=[float(x) for x in shifts_raw],
                    note="control variate averaged over its %d exact-set positions against the FP64 energies "
                         "of the same %d walkers (clipped to the median -+ sqrt(2/dt)); split-BF16 against FP64 "
                         "propagation from the trial with identical fields, block energy per step"
                         % (subset_inv, W))
    finally:
        for c in ctx:
            c.close()


def cpu_baseline(ham, spec, threads):
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_lib as O
    orc = O.Oracle(ham, threads, spec["walker_rhf"])
    orc.prep_prop(ham.phi_up, ham.phi_dn, spec["dt"])
    d = ham.serial_det(ham.phi_up, ham.phi_dn)
    orc.set_walkers(np.tile(d, (threads, 1)))
    nsteps = max(1, int(os.environ.get("AFQ_CPU_STEPS", "8")))
    rate, secs = orc.bench(threads, nsteps, 1, spec["ortho"], 7)
    return dict(value=rate, unit="walker-steps/s", cores=threads, kind="port",
                nproc=os.cpu_count(), cores_note="threads = the host cores this job may use, at most the "
                "box's 16-core share of the node for one GPU",
                sample="%d walkers x %d steps (same workload), E_L every step, QR every %d, "
                       "%.1f s on %d host threads (oracle/afqmc_oracle.cpp)"
                       % (threads, nsteps, spec["ortho"], secs, threads))


def micro(kind, workload, nwalk=1024, calls=8, chunks=None, variants64=None, variants=None):
    """Kernel microbenchmark for profiling: one context of `nwalk` walkers near the
    trial, `calls` measurements with the exchange in the given precision."""
    from vmc_amd.abi import AFQ_PREC_BF16, AFQ_PREC_BF16X3, AFQ_PREC_FP64, AFQ_PREC_FP8
    from vmc_amd.afqmc import Context
    from vmc_amd.synthetic import workload as get_workload
    prec = {"exchange-bf16": AFQ_PREC_BF16, "exchange-bf16x3": AFQ_PREC_BF16X3, "exchange-fp64": AFQ_PREC_FP64,
            "exchange-fp8": AFQ_PREC_FP8, "prop-split": AFQ_PREC_BF16X3, "vhs-split": AFQ_PREC_BF16X3,
            "fb-split": AFQ_PREC_BF16X3}[kind]
    h, spec = get_workload(workload)
    if kind in ("prop-split", "vhs-split", "fb-split"):
        nwalk = spec["nwalk"]
    ctx = Context(h, nwalk, spec["walker_rhf"])
    ctx.prep_prop(h.phi_up, h.phi_dn, spec["dt"])
    rng = np.random.default_rng(0)
    dets = []
    for _ in range(nwalk):
        up = h.phi_up + 0.02 * (rng.standard_normal(h.phi_up.shape) + 1j * rng.standard_normal(h.phi_up.shape))
        dn = h.phi_dn + 0.02 * (rng.standard_normal(h.phi_dn.shape) + 1j * rng.standard_normal(h.phi_dn.shape))
        dets.append(h.serial_det(up, dn))
    ctx.set_walkers(np.array(dets))
    if kind == "vhs-split":
        # the split-BF16 VHS tiles on the workload's population, one propagation each
        ctx.set_precision(prec_fb=prec, prec_vhs=prec)
        ctx.set_prop_precision(prec)
        for tile in (variants or [0, 1, 2, 3, 4]):
            ctx.set_vhs_tile(tile)
            ctx.set_walkers(np.array(dets))
            ctx.propagate(rng.standard_normal((nwalk, h.nchol)), 0.0)
            ctx.sync()
            ctx.stage_times(reset=True)
            for _ in range(calls):
                ctx.set_walkers(np.array(dets))
                ctx.propagate(rng.standard_normal((nwalk, h.nchol)), 0.0)
            ctx.sync()
            st = ctx.stage_times(reset=True)
            print(json.dumps({"micro": kind, "workload": workload, "nwalk": nwalk, "vhs_tile": tile,
                              "vhs_ms": st["vhs"] / calls}), flush=True)
        return
    if kind == "fb-split":
        # the split-BF16 force bias variants on the workload's population (each
        # set_walkers recomputes the Green's function and the force bias)
        ctx.set_precision(prec_fb=prec)
        for v in (variants or [0, 1]):
            ctx.set_force_bias_variant(v)
            ctx.set_walkers(np.array(dets))
            ctx.sync()
            ctx.stage_times(reset=True)
            for _ in range(calls):
                ctx.set_walkers(np.array(dets))
            ctx.sync()
            st = ctx.stage_times(reset=True)
            print(json.dumps({"micro": kind, "workload": workload, "nwalk": nwalk, "variant": v,
                              "force_bias_ms": st["force_bias"] / calls}), flush=True)
        return
    if kind == "prop-split":
        # the split propagation variants, timed by the autotuner on these walkers (it
        # writes to scratch, so every call sees the same walkers and V)
        from vmc_amd.afqmc import lib
        import ctypes as C
        ctx.set_precision(prec_fb=prec, prec_vhs=prec)
        ctx.set_prop_precision(prec)
        ctx.propagate(rng.standard_normal((nwalk, h.nchol)), 0.0)
        ctx.set_walkers(np.array(dets))
        out = []
        for _ in range(calls):
            ch, ms3 = C.c_int32(0), (C.c_double * 3)()
            assert lib().afq_autotune(ctx.ptr, C.byref(ch), ms3) == 0
            out.append(list(ms3))
        print(json.dumps({"micro": kind, "workload": workload, "nwalk": nwalk,
                          "ms_per_propagation": np.mean(out, axis=0).tolist()}))
        return
    ctx.set_precision(prec_exchange=prec)
    runs = [(ch, 0, v) for ch in (chunks or [0]) for v in (variants or [0])]
    if variants64:
        runs = [(0, v, 0) for v in variants64]
    for ch, v64, vx in runs:
        ctx.set_exchange_chunks(ch)
        ctx.set_exchange64_variant(v64)
        if kind == "exchange-bf16x3":
            ctx.set_exchange3_variant(vx)   # 0 pair-wise, 1 tiled
        else:
            ctx.set_exchange_variant(vx)
        ctx.measure()
        ctx.sync()
        ctx.stage_times(reset=True)
        t0 = time.time()
        for _ in range(calls):
            ctx.measure()
        ctx.sync()
        ms = (time.time() - t0) / calls * 1e3
        st = ctx.stage_times(reset=True)
        print(json.dumps({"micro": kind, "workload": workload, "nwalk": nwalk, "chunks": ch, "fp64_variant": v64,
                          "variant": vx,
                          "ms_per_measure": ms,
                          "exchange_ms": st["exchange"] / calls,
                          "tflops": exchange_flops(spec, nwalk) / (st["exchange"] / calls * 1e-3) / 1e12}),
              flush=True)


def bench_batched(a):
    """The uneven multi-system workload: 64 systems, N ~ U{20..120}, n = round(N/5),
    G = 4N, 256 walkers each; every step of every system is one hipGraph launch whose
    kernels are grouped (one launch per stage and kernel for all systems), against the
    same step with one graph branch per system and with the systems grouped on 4 streams.
    Walker-steps count the walkers each system propagated (weight > 1e-8 at the step's
    start); the FLOP rate counts those propagations plus the measurements of the walkers
    alive after them."""
    from vmc_amd.synthetic import batched_systems
    t0 = time.time()
    hams = batched_systems()  # worker processes: before any GPU call in this process
    log = lambda *x: print(*x, file=sys.stderr, flush=True)  # noqa: E731
    log("[bench] %d systems built in %.1fs" % (len(hams), time.time() - t0))
    from vmc_amd.abi import AFQ_PREC_BF16X3
    from vmc_amd.afqmc import Batch
    W, dt, ortho = 256, 0.005, 5
    half = np.sqrt(2.0 / dt)
    parts = [split_flops(dict(norb=h.norb, nchol=h.nchol, nalpha=h.nalpha, nbeta=h.nbeta, walker_rhf=False), ortho)
             for h in hams]
    paths, first = {}, {}
    for name, mixed, graph, lanes in (("fp64_eager", False, False, 1), ("fp64_branches", False, True, 0),
                                      ("fp64_graph", False, True, 1), ("mixed_branches", True, True, 0),
                                      ("mixed_graph_4lanes", True, True, 4), ("mixed_graph", True, True, 1)):
        b = Batch(hams, False, W)
        b.set_lanes(lanes)
        et = np.zeros(len(hams))
        for i, (c, h) in enumerate(zip(b.ctx, hams)):
            c.prep_prop(h.phi_up, h.phi_dn, dt)
            o = c.ham_and_overlap(h.serial_det(h.phi_up, h.phi_dn)[None, :], h.nchol)[0]
            et[i] = (o[0] / o[1]).real
            c.set_walkers(np.tile(h.serial_det(h.phi_up, h.phi_dn), (W, 1)))
            if mixed:
                c.set_precision(prec_fb=AFQ_PREC_BF16X3, prec_vhs=AFQ_PREC_BF16X3, prec_exchange=AFQ_PREC_BF16X3)
                c.set_prop_precision(AFQ_PREC_BF16X3)
        tune = b.autotune()
        b.capture(20261202, ortho, half, first_step=1)
        nlaunch = (b.launches(False), b.launches(True))
        eshift, eest, center = et.copy(), et.copy(), et.copy()
        rng = np.random.default_rng(5)
        total = a.warmup + a.steps
        tstart = None
        nprop, nlive = 0, 0
        work = collections.Counter()
        for step in range(1, total + 1):
            if step == a.warmup + 1:
                tstart = time.time()
            tot = b.step(step, eshift, rng.uniform(size=len(hams)), center, graph=graph)
            prop, live = b.counts()
            if step > a.warmup:
                nprop += int(prop.sum())
                nlive += int(live.sum())
                for p, ni, nl in zip(parts, prop, live):
                    for (part, prec), f in p.items():
                        work[prec if mixed else "fp64"] += f * (ni if part == "prop" else nl)
            eb = tot[:, 1] / tot[:, 0]
            if step == 1:
                first[name] = eb.copy()
            eest = 0.9 * eest + 0.1 * eb
            eshift = eest - 0.1 * np.log(tot[:, 0] / W) / dt
            center = eest
        wall = time.time() - tstart
        b.close()
        ms = 1e3 * wall / a.steps
        flops = sum(work.values())
        # the precision-weighted peak: three BF16 passes per split product
        tpk = work["bf16x3"] * 3 / PEAKS["bf16"] + work["fp64"] / PEAKS["fp64"]
        paths[name] = dict(walker_steps_per_s=nprop / wall, ms_per_step=ms,
                           propagated_per_step=nprop / a.steps, measured_per_step=nlive / a.steps,
                           step_tflops_algorithmic=flops / wall / 1e12,
                           peak_precision_weighted=flops / tpk if tpk else None,
                           launches_per_step=None if nlaunch[0] < 0 else {"plain": nlaunch[0], "qr": nlaunch[1]},
                           form="grouped on %d stream(s)" % lanes if lanes else "one graph branch per system",
                           taylor_tiles={"64x128": sum(1 for ch, _ in tune if ch == 1),
                                         "128x128c": sum(1 for ch, _ in tune if ch == 2)})
        log("[bench] %s: %.1f walker-steps/s, %.2f ms/step, per step %.0f propagated / %.0f measured"
            % (name, paths[name]["walker_steps_per_s"], ms, nprop / a.steps, nlive / a.steps))
    rel = float(np.max(np.abs(first["mixed_graph"] - first["fp64_graph"]) / np.abs(first["fp64_graph"])))
    best = paths["mixed_graph"]
    ach, pk = best["step_tflops_algorithmic"], best["peak_precision_weighted"]
    if ach > pk:
        log("[bench] refusing to print: %.1f TFLOP/s exceeds the precision-weighted peak %.1f" % (ach, pk))
        sys.exit(3)
    out = {
        "metric": METRIC, "value": best["walker_steps_per_s"], "unit": "walker-steps/s", "n_gpus": 1,
        "steps": a.steps, "warmup": a.warmup, "ms_per_step": best["ms_per_step"], "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64+bf16", "data": "synthetic",
        "config": {"workload": "%d systems, N ~ U{20..120} (sum %d), n = round(N/5), G = 4N, UHF trials, Cholesky "
                               "entries N(0, 0.3^2/N), %d walkers each, dt=%g, E_L every step, QR every %d, one "
                               "hipGraph launch per step of grouped kernels (one launch per stage and kernel for all "
                               "systems); throughput counts the walkers propagated"
                               % (len(hams), sum(h.norb for h in hams), W, dt, ortho),
                   "name": "c2", "path": "mixed_graph"},
        "roofline": {"bound": "mfma", "achieved": ach, "peak": pk, "unit": "TFLOP/s",
                     "frac": ach / pk, "traffic": None, "kernel": "whole step, all systems",
                     "note": "algorithmic FLOPs of every system's step (walkers propagated, walkers measured) over "
                             "the precision-weighted peak (split-BF16 products at a third of the BF16 peak, the "
                             "rest at the FP64 peak)"},
        "cpu_baseline": None,
        "paths": paths,
        "speedup_vs_fp64_graph": best["walker_steps_per_s"] / paths["fp64_graph"]["walker_steps_per_s"],
        "grouped_vs_branches_mixed": best["walker_steps_per_s"] / paths["mixed_branches"]["walker_steps_per_s"],
        "grouped_vs_branches_fp64": paths["fp64_graph"]["walker_steps_per_s"]
        / paths["fp64_branches"]["walker_steps_per_s"],
        "graph_speedup_fp64": paths["fp64_graph"]["walker_steps_per_s"] / paths["fp64_eager"]["walker_steps_per_s"],
        "first_step_energy_rel_diff_mixed_vs_fp64": rel,
    }
    print(json.dumps(out))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--workload", default="c4")
    ap.add_argument("--train-steps", type=int, default=0,
                    help="exact FP64 steps whose (walker, E_K - E_J) pairs train the surrogate "
                         "(default: ~48k pairs)")
    ap.add_argument("--epochs", type=int, default=20)
    ap.add_argument("--subset-inv", type=int, default=16)
    ap.add_argument("--risk-frac", type=float, default=0.05,
                    help="learned-surrogate path: fraction of live walkers (largest |E_J - median|) "
                         "always measured exactly")
    ap.add_argument("--fp64-only", action="store_true")
    ap.add_argument("--no-mlp", action="store_true", help="skip the learned-surrogate path")
    ap.add_argument("--mlp", action="store_true",
                    help="(the learned-surrogate path runs by default; kept for old command lines)")
    ap.add_argument("--surrogate-prec", choices=["bf16", "bf16x3", "fp8"], default="bf16",
                    help="precision of the exchange surrogate level of the control variate")
    ap.add_argument("--exact-prec", choices=["fp64", "bf16x3"], default="bf16x3",
                    help="exchange precision of the control variate's exact level (the subset): split BF16 with "
                         "three MFMA passes (default; about FP32 accurate, its shift against FP64 is measured on "
                         "every walker of the workload and printed), or FP64")
    ap.add_argument("--fp64-propagation", action="store_true",
                    help="mixed path: keep the force bias, VHS and Taylor products in FP64 "
                         "(default: split BF16)")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-shift-check", action="store_true",
                    help="skip the deterministic energy-shift checks (control-variate expectation, split "
                         "propagation on identical walkers)")
    ap.add_argument("--cpu-threads", type=int, default=0)
    ap.add_argument("--calibrate", action="store_true",
                    help="also run the 1 GiB plain-copy kernel (HBM counter calibration)")
    ap.add_argument("--micro", choices=["exchange-bf16", "exchange-bf16x3", "exchange-fp64", "exchange-fp8",
                                        "prop-split", "vhs-split", "fb-split"],
                    help="kernel microbenchmark for profiling instead of the bench: an exchange precision "
                         "(1024 walkers, 8 measurements), or prop-split (the split propagation variants "
                         "on the workload's walkers, 8 autotuner rounds), vhs-split (the split VHS tiles) or "
                         "fb-split (the split force bias variants)")
    ap.add_argument("--micro-walkers", type=int, default=1024)
    ap.add_argument("--xc64-variants", default="",
                    help="microbenchmark: comma-separated FP64 exchange kernels to time (0, 1, 2)")
    ap.add_argument("--xc-variants", default="",
                    help="microbenchmark: comma-separated one-pass BF16 exchange kernels to time (0 .. 3)")
    ap.add_argument("--xc-chunks", default="",
                    help="microbenchmark: comma-separated chunk counts of the pair-wise exchange to time")
    a = ap.parse_args()
    if a.micro:
        if a.calibrate:
            from vmc_amd.afqmc import debug_copy
            debug_copy(1 << 30)
        micro(a.micro, a.workload, nwalk=a.micro_walkers,
              chunks=[int(x) for x in a.xc_chunks.split(",")] if a.xc_chunks else None,
              variants64=[int(x) for x in a.xc64_variants.split(",")] if a.xc64_variants else None,
              variants=[int(x) for x in a.xc_variants.split(",")] if a.xc_variants else None)
        return
    if a.workload == "c2":
        if a.gpus != 1:
            print("bench.py: this build runs on one GPU; --gpus %d is not supported" % a.gpus, file=sys.stderr)
            sys.exit(2)
        bench_batched(a)
        return
    if a.gpus != 1:
        print("bench.py: this build runs one GPU holding one rank's walker population; "
              "--gpus %d is not supported" % a.gpus,
              file=sys.stderr)
        sys.exit(2)
    from vmc_amd.abi import (AFQ_ENERGY_SURROGATE, AFQ_PREC_BF16, AFQ_PREC_BF16X3, AFQ_PREC_FP64, AFQ_PREC_FP8,
                             AFQ_SURR_EXCHANGE,
                             AFQ_SURR_MLP)
    from vmc_amd.synthetic import workload
    t0 = time.time()
    ham, spec = workload(a.workload)
    W = spec["nwalk"]
    print("[bench] workload %s built in %.1fs" % (a.workload, time.time() - t0), file=sys.stderr, flush=True)
    if a.calibrate:
        from vmc_amd.afqmc import debug_copy
        debug_copy(1 << 30)
    T = a.train_steps or max(2, (48 * 1024 + W - 1) // W)
    log = lambda *x: print(*x, file=sys.stderr, flush=True)  # noqa: E731
    paths = {}
    fp64 = run_path(ham, spec, a.warmup + a.steps, a.warmup)
    # the exchange runs on the live walkers only (dead walkers get no local energy)
    fp64.update(exchange_prec="fp64", n_exact=fp64["measured_per_step"])
    paths["fp64"] = fp64
    log("[bench] fp64: %.1f walker-steps/s, %.1f ms/step, per step %.1f propagated / %.1f measured, %d restarts"
        % (fp64["walker_steps_per_s"], fp64["ms_per_step"], fp64["propagated_per_step"], fp64["measured_per_step"],
           fp64["restarts"]))
    best_name = "fp64"
    if not a.fp64_only:
        # surrogate = the exchange in one BF16 pass on every walker; exact FP64 on a
        # random 1/subset_inv of the walkers (Horvitz-Thompson correction)
        pp = AFQ_PREC_FP64 if a.fp64_propagation else AFQ_PREC_BF16X3
        xprec = {"fp64": AFQ_PREC_FP64, "bf16x3": AFQ_PREC_BF16X3}[a.exact_prec]
        xcv = run_path(ham, spec, a.warmup + a.steps, a.warmup, energy_mode=AFQ_ENERGY_SURROGATE,
                       prec_fb=pp, prec_vhs=pp, prec_prop=pp, prec_exchange=xprec,
                       surrogate_kind=AFQ_SURR_EXCHANGE,
                       surrogate_prec={"bf16": AFQ_PREC_BF16, "bf16x3": AFQ_PREC_BF16X3,
                                       "fp8": AFQ_PREC_FP8}[a.surrogate_prec],
                       subset_inv=a.subset_inv, risk_frac=0.0, shadow_exact=True)
        xcv.update(exchange_prec=a.exact_prec, surrogate_prec=a.surrogate_prec, n_exact=xcv["exact_per_step"],
                   fb_vhs_prec="fp64" if a.fp64_propagation else "bf16x3")
        xcv.update(cv_summary(xcv, fp64))
        paths["mixed_exchange_cv"] = xcv
        log("[bench] mixed (%s exchange level + %s 1/%d subset): %.1f walker-steps/s, %.1f ms/step, "
            "speedup %.2fx, sampled shift %.4f +- %s mHa, err/sqrt(s) ratio %s, per step %.1f propagated / "
            "%.1f measured / %.1f exact"
            % (a.surrogate_prec, a.exact_prec, a.subset_inv, xcv["walker_steps_per_s"], xcv["ms_per_step"], xcv["speedup_vs_fp64"],
               xcv["energy_shift_mha"], xcv["energy_shift_sem_mha"], xcv["err_per_sqrt_s_ratio"],
               xcv["propagated_per_step"], xcv["measured_per_step"], xcv["exact_per_step"]))
        best_name = "mixed_exchange_cv"
        if not a.no_mlp:
            mlp = run_path(ham, spec, T + a.warmup + a.steps, T + a.warmup, energy_mode=AFQ_ENERGY_SURROGATE,
                           prec_exchange=AFQ_PREC_FP64, surrogate_kind=AFQ_SURR_MLP, surrogate_train_steps=T,
                           surrogate_hidden=256, surrogate_epochs=a.epochs, subset_inv=a.subset_inv,
                           risk_frac=a.risk_frac, shadow_exact=True)
            mlp.update(exchange_prec="fp64", n_exact=mlp["exact_per_step"], surrogate="mlp")
            mlp.update(cv_summary(mlp, fp64))
            paths["mlp_cv"] = mlp
            log("[bench] mlp surrogate (train rmse %.3g, valid %.3g Ha): %.1f walker-steps/s, %.1f ms/step, "
                "speedup %.2fx, shift %.4f +- %s mHa, err/sqrt(s) ratio %s, live %.3f"
                % (mlp["train_rmse"], mlp["valid_rmse"], mlp["walker_steps_per_s"], mlp["ms_per_step"],
                   mlp["speedup_vs_fp64"], mlp["energy_shift_mha"], mlp["energy_shift_sem_mha"],
                   mlp["err_per_sqrt_s_ratio"], mlp["live_frac"]))
    for name, pth in paths.items():
        pth["rooflines"] = stage_rooflines(spec, pth, pth["n_exact"])
    best = paths[best_name]
    # the dominant kernel: largest share of the step
    shares = {k: best["stage_ms_per_step"][k] for k in best["rooflines"]}
    dom_name = max(shares, key=shares.get)
    dom = dict(best["rooflines"][dom_name])
    dom["stage"] = dom_name
    dom["traffic"] = profiled_traffic(a.workload, dom.get("profile_row", dom.get("symbol")))
    if dom["traffic"] is not None:
        dom["traffic_source"] = os.path.relpath(PROFILE_HBM, ROOT)
    cpu = None
    if not a.no_cpu:
        threads = a.cpu_threads or host_cores()
        cpu = cpu_baseline(ham, spec, threads)
        log("[bench] cpu baseline: %.2f walker-steps/s on %d threads" % (cpu["value"], threads))
    wstep = flops_per_walker_step(spec)
    wprop = flops_per_walker_step(spec, energy=False)
    for name, pth in paths.items():
        pth.pop("energies", None)
        pth.pop("weights", None)
        # useful work of a step: every propagated walker's step and every measured walker's E_L
        # (the learned surrogate evaluates the exchange on the exact subset only, and its
        # network in place of it on the others)
        step_flops = wprop * pth["propagated_per_step"] + (wstep - wprop) * pth["measured_per_step"]
        if pth.get("surrogate") == "mlp":
            F = spec["nchol"] + 2 * spec["norb"]
            mlp_flops = 2.0 * (F * 256 + 2 * 256 * 256 + 256)
            xw = exchange_flops(spec, 1)
            step_flops += (pth["n_exact"] - pth["measured_per_step"]) * xw + pth["measured_per_step"] * mlp_flops
        pth["step_tflops_algorithmic"] = step_flops / (pth["ms_per_step"] * 1e-3) / 1e12
        pth["peak_precision_weighted"] = precision_weighted_peak(pth["rooflines"])
        bad = [k for k, r in pth["rooflines"].items() if r["frac"] > 1.0]
        if bad or pth["step_tflops_algorithmic"] > pth["peak_precision_weighted"]:
            print("bench.py: %s path: a stage or the step exceeds its peak (%s; step %.1f TFLOP/s against a "
                  "precision-weighted peak of %.1f): the work counts are wrong, no line printed"
                  % (name, bad, pth["step_tflops_algorithmic"], pth["peak_precision_weighted"]), file=sys.stderr)
            sys.exit(3)
    shift = None
    if best_name != "fp64" and not a.no_shift_check:
        shift = deterministic_shift(ham, spec, a.subset_inv, {"fp64": AFQ_PREC_FP64, "bf16x3": AFQ_PREC_BF16X3}[
            a.exact_prec])
        log("[bench] cv expectation residual %.3e mHa (unclipped %.3e); split propagation block shift %s mHa "
            "(unclipped %s); clipped fraction %.3f"
            % (shift["cv_expectation_residual_mha"], shift["cv_expectation_unclipped_residual_mha"],
               shift["propagation_shift_mha"], shift["propagation_unclipped_shift_mha"], shift["clipped_fraction"]))
    out = {
        "metric": METRIC,
        "value": best["walker_steps_per_s"],
        "unit": "walker-steps/s",
        "n_gpus": 1,
        "steps": best["steps"],
        "warmup": a.warmup,
        "ms_per_step": best["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64" if best_name == "fp64" else "f64+bf16",
        "data": "synthetic",
        "config": {"workload": "N=%d %da+%db G=%d %s trial, Cholesky entries N(0, %s), %d walkers, dt=%g, E_L and "
                               "comb every step, QR every %d; the population restarts at the trial every %d steps "
                               "outside the timings; throughput counts the walkers propagated"
                   % (spec["norb"], spec["nalpha"], spec["nbeta"], spec["nchol"], spec["trial"].upper(),
                      "0.3^2/N" if spec.get("coupling") is None else "(%g/N)^2" % spec["coupling"],
                      W, spec["dt"], spec["ortho"], RESTART_EVERY),
                   "name": a.workload, "path": best_name, "subset_inv": a.subset_inv},
        "roofline": dom,
        "cpu_baseline": cpu,
        "paths": paths,
        "flops_per_walker_step": wstep,
    }
    if best_name != "fp64":
        out["speedup_vs_fp64"] = best["speedup_vs_fp64"]
        out["err_per_sqrt_s_ratio"] = best["err_per_sqrt_s_ratio"]
        # the shift in the metric: the control variate's expectation against the FP64
        # energies of the same walkers (zero up to round-off) and the block-energy change the
        # split-BF16 propagation makes on identical walkers and fields
        if shift is not None:
            out["energy_shift_mha"] = shift["cv_expectation_residual_mha"]
            out["energy_shift_unclipped_mha"] = shift["cv_expectation_unclipped_residual_mha"]
            out["energy_shift_check"] = shift
        out["energy_shift_sampled_mha"] = best["energy_shift_mha"]
        out["energy_shift_sampled_sem_mha"] = best["energy_shift_sem_mha"]
        out["energy_shift_sampled_blocks"] = best["energy_shift_blocks"]
    print(json.dumps(out))


if __name__ == "__main__":
    main()
