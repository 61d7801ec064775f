"""The FP64 exchange kernel at the edges of its tiles (64 rows and columns of whole vectors and
walkers) against a numpy evaluation, with dead walkers, a short last chunk of vectors and a
truncated vector count.

E_K = 1/2 sum_s m_s Re sum_g sum_ij f_ij f_ji, f = R_sg theta_s: each f is an FP64 sum of N products
and a thread adds a few hundred pairs, so the error is at most (2 N + 1000) 2^-53 (1.4e-13) of the sum
of magnitudes, and theta is good to a few 1e-15: 1e-12 of that sum bounds it."""
import numpy as np
import pytest

from vmc_amd.abi import HamArrays
from vmc_amd.afqmc import Context

pytestmark = pytest.mark.gpu

CASES = [
    # N, na, nb, G, W, vectors in the energy
    (5, 3, 3, 7, 5, 7),          # below the kernel's smallest n: the other kernel
    (6, 4, 4, 33, 40, 33),       # 16 x 16 blocks, one thread each; more than two row tiles of vectors
    (11, 5, 4, 40, 13, 27),      # slots of different size, a truncated vector count
    (21, 13, 13, 64, 9, 64),     # odd n, one walker past a tile, N of one K step past a multiple of 4
    (30, 16, 16, 50, 7, 50),     # the tile full
    (23, 17, 17, 31, 4, 31),     # 51 rows: the second half as two tiles; odd
    (40, 22, 21, 45, 6, 20),     # 44 and 42 rows: the second half as one tile
    (34, 32, 31, 21, 3, 21),
    (36, 33, 33, 17, 3, 17),     # one walker and vector a tile, 33 rows
    (50, 47, 43, 9, 2, 9),
    (66, 64, 64, 10, 2, 10),     # the largest n
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "N%d_%d_%d_G%d_W%d" % c[:5])
def test_exchange_matches_numpy(case):
    N, na, nb, G, W, keep = case
    rng = np.random.default_rng(N)
    L = rng.standard_normal((G, N, N)) / N
    L = L + np.swapaxes(L, 1, 2)
    h1 = rng.standard_normal((N, N))
    h1 = h1 + h1.T
    phi = [np.linalg.qr(rng.standard_normal((N, n)))[0] for n in (na, nb)]
    h = HamArrays(N, na, nb, 0.0, h1, h1, L, phi[0], phi[1])
    dets = [[p + 0.1 * (rng.standard_normal(p.shape) + 1j * rng.standard_normal(p.shape)) for p in phi] for _ in range(W)]
    weights = np.ones(W)
    weights[W // 2] = 0.0
    ctx = Context(h, W, False)
    ctx.set_nchol_ene(keep)
    ctx.set_walkers(np.array([h.serial_det(*d) for d in dets]), weights=weights)
    ctx.measure()
    ek = ctx.energy_parts()[1]
    ctx.close()
    for w in np.flatnonzero(weights):
        ref = mag = 0.0
        for s in range(2):
            th = dets[w][s] @ np.linalg.inv(phi[s].T @ dets[w][s])
            R = np.einsum("mi,gmk->gik", phi[s], L[:keep])
            f = R @ th
            ref += 0.5 * np.einsum("gij,gji->", f, f).real
            a = np.abs(R) @ np.abs(th)
            mag += 0.5 * np.einsum("gij,gji->", a, a)
        assert abs(ek[w] - ref) <= 1e-12 * mag
    assert ek[W // 2] == 0.0


@pytest.mark.parametrize("case", [
    # at most 48 rows and columns: three waves a workgroup
    (40, 22, 22, 45, 7, 20), (41, 23, 23, 30, 4, 30), (24, 24, 24, 9, 3, 9), (33, 33, 33, 19, 3, 19), (49, 48, 48, 11, 2, 11),
], ids=lambda c: "N%d_%d_%d_G%d_W%d" % c[:5])
def test_exchange_three_waves_matches_numpy(case):
    test_exchange_matches_numpy(case)


@pytest.mark.parametrize("case", [
    # slots of one to three electrons, on both sides of a 128-row tile of vectors and walkers
    (4, 1, 1, 129, 130, 129), (7, 2, 1, 65, 129, 60), (9, 2, 2, 64, 64, 64), (10, 3, 2, 43, 43, 42), (10, 3, 3, 85, 90, 85),
], ids=lambda c: "N%d_%d_%d_G%d_W%d" % c[:5])
def test_exchange_of_few_electrons_matches_numpy(case):
    test_exchange_matches_numpy(case)
