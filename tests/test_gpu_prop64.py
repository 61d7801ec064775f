"""The fused FP64 propagation kernel against the separate one-body and Taylor kernels, at the
edges of its row tiles (16 and 64 orbitals), column blocks and LDS capacity, for restricted
and unrestricted integrals.

Seven products of at most 2N terms each round to at most 7 * 2N * 2^-53 of the orbitals'
scale (6e-13 at N = 384), in either order of summation: 2e-12 bounds the difference of two."""
import ctypes as C

import numpy as np
import pytest

from vmc_amd.abi import HamArrays
from vmc_amd.afqmc import Context, lib

pytestmark = pytest.mark.gpu

CASES = [
    # N, na, nb, unrestricted, RHF walker
    (3, 1, 1, False, True),        # one row tile, one electron
    (16, 8, 8, False, True),       # a full row tile, one full column tile
    (17, 5, 4, False, False),      # one row past the tile, two determinants in one tile
    (64, 21, 20, False, False),    # a wave's row tile each, six column tiles in two blocks
    (65, 9, 7, True, False),       # two row tiles for one wave; a block per spin
    (96, 40, 3, True, False),      # spins of very different width
    (128, 20, 20, False, False),   # five column tiles in one block
    (129, 24, 16, False, False),
    (193, 12, 12, False, False),
    (256, 17, 16, False, False),   # the largest N of five-tile blocks
    (257, 33, 31, False, False),
    (320, 64, 64, False, False),   # LDS full: 320 orbitals x 64 real columns
    (321, 25, 24, False, False),
    (384, 24, 24, False, False),   # the largest N
]


def set_variant(ctx, v):
    lib().afq_set_taylor_variant.argtypes = [C.c_void_p, C.c_int32]
    return lib().afq_set_taylor_variant(ctx.ptr, v)


def system(N, na, nb, unrestricted, seed):
    rng = np.random.default_rng(seed)
    G = 6

    def sym(a):
        return 0.5 * (a + np.swapaxes(a, -1, -2))

    L = [sym(rng.standard_normal((G, N, N))) / N for _ in range(2)]
    h = [sym(rng.standard_normal((N, N))) / N + np.diag(np.linspace(-2.0, 0.0, N)) for _ in range(2)]
    mod = [a - 0.5 * np.einsum("gij,gjk->ik", b, b) for a, b in zip(h, L)]
    phi = [np.linalg.qr(rng.standard_normal((N, n)))[0] for n in (na, nb)]
    more = dict(h1_dn=h[1], h1_mod_dn=mod[1], chol_dn=L[1]) if unrestricted else {}
    return HamArrays(N, na, nb, 0.0, h[0], mod[0], L[0], phi[0], phi[1], **more)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "N%d_%d_%d%s" % (c[0], c[1], c[2], "_u" if c[3] else ""))
def test_fused_matches_separate_kernels(case):
    N, na, nb, unrestricted, rhf = case
    h = system(N, na, nb, unrestricted, seed=N)
    if rhf:
        h = HamArrays(N, na, nb, 0.0, h.h1, h.h1_mod, h.chol, h.phi_up, trial_rhf=True)
    W = 3
    rng = np.random.default_rng(N + 1)

    def walker():
        up, dn = (p + 0.05 * (rng.standard_normal(p.shape) + 1j * rng.standard_normal(p.shape)) for p in (h.phi_up, h.phi_dn))
        return h.serial_det(up, up if rhf else dn)

    dets = np.array([walker() for _ in range(W)])
    draws = rng.standard_normal((W, h.nchol))
    out = []
    for variant in (0, 1, 2):
        ctx = Context(h, W, rhf)
        assert set_variant(ctx, variant) == 0
        ctx.prep_prop(h.phi_up, h.phi_dn, 0.01)
        ctx.set_walkers(dets, weights=np.array([1.0, 0.0, 2.0]))
        ctx.propagate(draws, 0.0)
        out.append(ctx.get_walkers()[0])
        ctx.close()
    scale = np.max(np.abs(out[1]))
    assert np.max(np.abs(out[0] - out[1])) <= 2e-12 * scale
    assert np.max(np.abs(out[0] - out[2])) <= 2e-12 * scale
    assert np.array_equal(out[0][1], dets[1]) and not np.array_equal(out[0][0], dets[0])   # weight zero: not propagated
