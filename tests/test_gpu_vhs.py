"""One propagation at the edges of the FP64 VHS kernel's tiles (orbitals in blocks of 4 and pairs
of blocks, vectors in K steps of 4 and pipelines of 3 steps, walkers in 16s, 32s and 64s) and on
each of its tile shapes, against the CPU oracle: a wrong element of the matrix or a wrong walker
shows in the determinants at sqrt(dt) of its size.  The oracle and the device agree to 1e-10 of
the largest element, as over whole trajectories."""
import numpy as np
import pytest

import oracle_lib as O
from vmc_amd.abi import HamArrays
from vmc_amd.afqmc import Context

pytestmark = pytest.mark.gpu

CASES = [
    # N, G, W, unrestricted integrals
    (1, 1, 3, False), (2, 3, 2, True), (3, 4, 17, False), (4, 5, 16, True), (5, 8, 15, False), (7, 11, 33, True),
    (8, 12, 32, False), (9, 13, 31, False), (13, 9, 65, True), (16, 16, 64, False), (17, 17, 5, True), (33, 25, 18, False),
    (64, 2, 1000, False),     # 32 walkers by 32 columns a wave
    (100, 2, 1024, False),    # 32 walkers by 64 columns
    (99, 3, 500, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "N%d_G%d_W%d%s" % (*c[:3], "_u" if c[3] else ""))
def test_propagation_matches_oracle(case):
    N, G, W, unrestricted = case
    rng = np.random.default_rng(N + G)
    na, nb = max(1, N // 8), 1

    def sym(*shape):
        a = rng.standard_normal(shape)
        return 0.5 * (a + np.swapaxes(a, -1, -2))

    L = [sym(G, N, N) / N for _ in range(2)]
    h1 = [sym(N, N) / N + np.diag(np.linspace(-2.0, 0.0, N)) for _ in range(2)]
    mod = [a - 0.5 * np.einsum("gij,gjk->ik", b, b) for a, b in zip(h1, L)]
    phi = [np.linalg.qr(rng.standard_normal((N, n)))[0] for n in (na, nb)]
    more = dict(h1_dn=h1[1], h1_mod_dn=mod[1], chol_dn=L[1]) if unrestricted else {}
    h = HamArrays(N, na, nb, 0.0, h1[0], mod[0], L[0], phi[0], phi[1], **more)
    dets = np.array([h.serial_det(*(p + 0.05 * (rng.standard_normal(p.shape) + 1j * rng.standard_normal(p.shape)) for p in phi))
                     for _ in range(W)])
    weights = rng.uniform(0.5, 2.0, W)
    weights[W // 2] = 0.0
    draws = rng.standard_normal((W, G))
    ctx, orc = Context(h, W, False), O.Oracle(h, W, False)
    for c in (ctx, orc):
        c.prep_prop(phi[0], phi[1], 0.01)
        c.set_walkers(dets, weights=weights)
    ctx.propagate(draws, 0.0)
    orc.propagate(draws, 0.0, 100.0)
    got, want = ctx.get_walkers(), orc.get_walkers()
    ctx.close()
    kept = want[2] != 0.0
    assert np.max(np.abs(got[0][kept] - want[0][kept])) <= 1e-10 * np.max(np.abs(want[0][kept]))
    assert np.max(np.abs(got[2] - want[2])) <= 1e-10 * np.max(want[2])
