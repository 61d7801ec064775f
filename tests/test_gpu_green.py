"""Overlap, theta = psi (Phi^T psi)^-1 and its one-body partial at the edges of the kernels' tiles
(electrons in eights and sixteens, orbitals in fours and sixteens, columns past the last walker)
against numpy.  theta is read through the force bias (both parts), the 1-RDM and the one-body
energy.

S has a condition of about 10 here, so n cond 2^-53 (7e-14 at n = 64) and the sums over at most
N n products bound every quantity to well below 1e-11 of its sum of magnitudes."""
import numpy as np
import pytest

from vmc_amd.abi import HamArrays
from vmc_amd.afqmc import Context

pytestmark = pytest.mark.gpu

CASES = [
    # N, na, nb, W
    (1, 1, 1, 3), (4, 2, 1, 5), (17, 8, 7, 3), (16, 9, 8, 4), (33, 16, 17, 2), (31, 24, 15, 3),
    (50, 25, 32, 3), (64, 33, 31, 2), (65, 40, 41, 2), (66, 48, 49, 3), (70, 57, 56, 2), (80, 64, 63, 2), (130, 64, 1, 2),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "N%d_%d_%d_W%d" % c)
def test_green_matches_numpy(case):
    N, na, nb, W = case
    G = 5
    rng = np.random.default_rng(N + na)
    L = rng.standard_normal((G, N, N))
    L = L + np.swapaxes(L, 1, 2)
    h1 = rng.standard_normal((N, N))
    h1 = h1 + h1.T
    phi = [np.linalg.qr(rng.standard_normal((N, n)))[0] for n in (na, nb)]
    h = HamArrays(N, na, nb, 0.0, h1, h1, L, phi[0], phi[1])
    dets = [[p + 0.1 * (rng.standard_normal(p.shape) + 1j * rng.standard_normal(p.shape)) for p in phi] for _ in range(W)]
    weights = rng.uniform(0.5, 2.0, W)
    weights[0] = 0.0 if W > 2 else 1.0
    ctx = Context(h, W, False)
    ctx.set_walkers(np.array([h.serial_det(*d) for d in dets]), weights=weights)
    fb, ov = ctx.force_bias(), ctx.overlaps()
    ctx.rdm_reset()
    ctx.rdm_accumulate()
    rdm = ctx.one_rdm(False)[0]
    ctx.measure()
    e1 = ctx.energy_parts()[0]
    ctx.close()
    live = np.flatnonzero(weights)
    acc, mag = np.zeros((2, N, N)), np.zeros((2, N, N))
    for w in range(W):
        th = [d @ np.linalg.inv(p.T @ d) for p, d in zip(phi, dets[w])]
        o = np.prod([np.linalg.det(p.T @ d) for p, d in zip(phi, dets[w])])
        assert abs(ov[w] - o) <= 1e-11 * abs(o)
        if w not in live:
            continue
        ref = sum(np.einsum("mi,gmk,ki->g", p, L, t) for p, t in zip(phi, th))
        top = sum(np.einsum("mi,gmk,ki->g", np.abs(p), np.abs(L), np.abs(t)) for p, t in zip(phi, th))
        assert np.all(np.abs(fb[w] - ref) <= 1e-11 * top)
        assert abs(e1[w] - sum(np.sum(t.real * (h1 @ p)) for p, t in zip(phi, th))) <= 1e-11 * sum(
            np.sum(np.abs(t) * np.abs(h1 @ p)) for p, t in zip(phi, th))
        for s in range(2):
            acc[s] += weights[w] * phi[s] @ th[s].real.T
            mag[s] += weights[w] * np.abs(phi[s]) @ np.abs(th[s]).T
    assert np.all(np.abs(rdm - acc / weights.sum()) <= 1e-11 * mag / weights.sum())
