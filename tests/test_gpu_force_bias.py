"""The FP64 force bias kernel at the edges of its tiles and of its split over K, against a numpy evaluation.

fb_g = sum_s m_s sum_k theta_s[k] R_sg[k]: the error of an FP64 sum of K products is at most
K 2^-53 sum |theta R| (7e-13 of it at K = 6,240, and theta itself is good to a few 1e-15),
so 1e-12 of sum |theta R| bounds it."""
import numpy as np
import pytest

from vmc_amd.afqmc import Context
from vmc_amd.synthetic import make_system

pytestmark = pytest.mark.gpu

CASES = [
    # N, na, nb, G, trial, W
    (5, 2, 2, 9, "rhf", 1),          # K = 10: one partial stage, one walker
    (13, 5, 4, 63, "uhf", 33),       # odd K, G and 2W one off the tile
    (24, 7, 7, 65, "uhf", 16),       # K split into two chunks
    (51, 13, 11, 205, "uhf", 70),    # small tile, several chunks, the last one short
    (40, 8, 8, 160, "rhf", 700),     # large tile (66 of them), K = 320 in chunks
    (60, 52, 52, 129, "uhf", 800),   # large tile, K = 6,240
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "N%d_%d_%d_G%d_%s_W%d" % c)
def test_force_bias_matches_numpy(case):
    N, na, nb, G, trial, W = case
    h = make_system(N, na, nb, G, seed=7, trial=trial)
    rhf = trial == "rhf"
    rng = np.random.default_rng(N + W)
    dets = []
    for _ in range(W):
        up = h.phi_up + 0.1 * (rng.standard_normal((N, na)) + 1j * rng.standard_normal((N, na)))
        dn = up if rhf else h.phi_dn + 0.1 * (rng.standard_normal((N, nb)) + 1j * rng.standard_normal((N, nb)))
        dets.append((up, dn))
    weights = np.ones(W)
    weights[W // 2::5] = 0.0 if W > 4 else 1.0   # dead walkers among the live ones
    ctx = Context(h, W, rhf)
    ctx.set_walkers(np.array([h.serial_det(*d) for d in dets]), weights=weights)
    fb = ctx.force_bias()
    ctx.close()
    live = np.flatnonzero(weights)
    ref, mag = np.zeros((len(live), G), complex), np.zeros((len(live), G))
    for s, phi in enumerate((h.phi_up, h.phi_dn)):
        R = np.einsum("mi,gmk->gki", phi, h.chol).reshape(G, -1)
        th = np.stack([dets[w][s] @ np.linalg.inv(phi.T @ dets[w][s]) for w in live]).reshape(len(live), -1)
        ref += th @ R.T
        mag += np.abs(th) @ np.abs(R).T
    assert np.all(np.abs(fb[live] - ref) <= 1e-12 * mag)
