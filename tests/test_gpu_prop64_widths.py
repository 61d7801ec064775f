"""The fused FP64 propagation with every width of its column blocks that each number of row tiles allows,
whole and with a short last tile, one block and several, against the separate one-body and Taylor kernels.

A wide block is only taken by a population that fills the chip, so 256 walkers.  The bound is that of
test_gpu_prop64: seven products of at most 2N terms, each rounding to 7 * 2N * 2^-53 of the orbitals'
scale (6e-13 at N = 384) in either order of summation."""
import ctypes as C

import numpy as np
import pytest
from test_gpu_prop64 import set_variant, system

from vmc_amd.abi import HamArrays
from vmc_amd.afqmc import Context, lib

pytestmark = pytest.mark.gpu

W = 256


def width(N, na, nb, unrestricted, rhf):
    """(column tiles a block, blocks) that W walkers take: the least rounds of 256 workgroups times the
    width, the widest of equals."""
    t = [-(-na // 8), -(-nb // 8)] if unrestricted else [-(-(na if rhf else na + nb) // 8), 0]
    best = None
    for c in range(min(5 if N <= 256 else 4 if N <= 320 else 3, max(t)), 0, -1):
        blocks = sum(-(-x // c) for x in t)
        cost = -(-blocks * W // 256) * c
        if best is None or cost < best[0]:
            best = cost, c, blocks
    return best[1:]


LAST = {1: 40, 2: 128, 3: 150, 4: 256, 5: 320, 6: 380}   # orbitals for 1 .. 6 row tiles a wave
CASES = [(N, 4 * c, 4 * c - (0 if c % 2 else 3), False, False, c, 1) for m, N in LAST.items()
         for c in range(1, (5 if m <= 4 else 4 if m == 5 else 3) + 1)]
CASES += [
    # N, na, nb, unrestricted, RHF walker, width, blocks
    (64, 24, 23, False, False, 3, 2),      # two blocks
    (100, 40, 39, False, False, 5, 2),
    (256, 32, 29, False, False, 4, 2),
    (300, 64, 61, False, False, 4, 4),
    (384, 36, 33, False, False, 3, 3),
    (72, 31, 31, False, True, 4, 1),       # one determinant
    (256, 40, 40, False, True, 5, 1),
    (50, 16, 15, True, False, 2, 2),       # a block per spin, each with its own E and V
    (97, 31, 27, True, False, 4, 2),
    (160, 40, 39, True, False, 5, 2),
    (250, 24, 19, True, False, 3, 2),
    (320, 32, 30, True, False, 4, 2),
    (370, 24, 24, True, False, 3, 2),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "N%d_%d_%d%s%s_ct%d" % (c[0], c[1], c[2], "_u" if c[3] else "",
                                                                           "_rhf" if c[4] else "", c[5]))
def test_every_width_matches_separate_kernels(case):
    N, na, nb, unrestricted, rhf, ct, blocks = case
    assert width(N, na, nb, unrestricted, rhf) == (ct, blocks)
    h = system(N, na, nb, unrestricted, seed=N + ct)
    if rhf:
        h = HamArrays(N, na, nb, 0.0, h.h1, h.h1_mod, h.chol, h.phi_up, trial_rhf=True)
    rng = np.random.default_rng(N + na)
    phi = [h.phi_up, h.phi_up if rhf else h.phi_dn]
    parts = []
    for p in phi:
        z = rng.standard_normal((W,) + p.shape + (2,))
        parts.append((p + 0.05 * (z[..., 0] + 1j * z[..., 1])).reshape(W, -1))
    dets = np.concatenate([parts[0], parts[0] if rhf else parts[1]], axis=1)
    weights = np.ones(W)
    weights[[1, 100, W - 2]] = 0.0
    draws = rng.standard_normal((W, h.nchol))
    out = []
    for variant in (0, 1, 2):
        ctx = Context(h, W, rhf)
        assert set_variant(ctx, variant) == 0
        ctx.prep_prop(*phi, 0.01)
        ctx.set_walkers(dets, weights=weights)
        ctx.propagate(draws, 0.0)
        out.append(ctx.get_walkers()[0])
        ctx.close()
    scale = np.max(np.abs(out[1]))
    assert np.max(np.abs(out[0] - out[1])) <= 2e-12 * scale
    assert np.max(np.abs(out[0] - out[2])) <= 2e-12 * scale
    dead = weights == 0.0
    assert np.array_equal(out[0][dead], dets[dead]) and not np.any(np.all(out[0][~dead] == dets[~dead], axis=1))


def test_autotuner_times_whole_propagations():
    """Every variant is timed over the same work, both one-body factors included: against the stage timers of
    steps taken with it (the factors are a tenth of it or more, half of which the comparison asks for)."""
    h = system(100, 24, 20, False, seed=5)
    ctx = Context(h, 1024, False)
    ctx.prep_prop(h.phi_up, h.phi_dn, 0.01)
    ctx.set_walkers_uniform(h.serial_det(h.phi_up, h.phi_dn))
    stages = []
    for variant in (1, 2):
        assert set_variant(ctx, variant) == 0
        times = []
        for step in range(6):
            ctx.set_weights(np.ones(1024))
            ctx.stage_times()
            ctx.propagate(None, 0.0, seed=1, step=step)
            times.append([ctx.stage_times(reset=False)[k] for k in ("taylor", "onebody")])
        stages.append(np.median(times[1:], axis=0))
    ctx.set_weights(np.ones(1024))
    choice, ms = C.c_int32(0), (C.c_double * 3)()
    assert lib().afq_autotune(ctx.ptr, C.byref(choice), ms) == 0
    ctx.stage_times()
    ctx.propagate(None, 0.0, seed=1, step=9)
    kept = ctx.stage_times()
    ctx.close()
    print("whole propagations", list(ms), "taylor, one-body", stages, "kept", kept["taylor"] + kept["onebody"])
    for t, (taylor, onebody) in zip(ms, stages):
        assert t >= taylor + 0.5 * onebody
    assert kept["taylor"] + kept["onebody"] <= 1.1 * min(ms[0], ms[1])
