"""Overlap and S^-1 where a wave takes a whole matrix (more than 512 matrices of at most 32 electrons),
at the edges of its column counts, and where several share one, against numpy.  theta = psi S^-1 is
read through the force bias.

S has a condition of about 10, so n cond 2^-53 (4e-14 at n = 32) and the sums over at most N n
products bound both to well below 1e-11 of their sums of magnitudes."""
import numpy as np
import pytest

from vmc_amd.abi import HamArrays
from vmc_amd.afqmc import Context

pytestmark = pytest.mark.gpu

CASES = [(1, 8, 257), (9, 12, 257), (13, 16, 260), (17, 20, 257), (21, 24, 257), (25, 32, 257), (32, 31, 256), (16, 15, 256), (8, 33, 257)]


@pytest.mark.parametrize("na,nb,W", CASES)
def test_many_matrices(na, nb, W):
    N, G = max(na, nb) + 4, 3
    rng = np.random.default_rng(na)
    L = rng.standard_normal((G, N, N))
    L = L + np.swapaxes(L, 1, 2)
    phi = [np.linalg.qr(rng.standard_normal((N, n)))[0] for n in (na, nb)]
    h = HamArrays(N, na, nb, 0.0, np.eye(N), np.eye(N), L, phi[0], phi[1])
    psi = [p + 0.1 * (rng.standard_normal((W,) + p.shape) + 1j * rng.standard_normal((W,) + p.shape)) for p in phi]
    # rows in another order in every walker's overlap matrix: pivots off the diagonal
    psi = [np.stack([x[:, rng.permutation(x.shape[1])] for x in p]) for p in psi]
    ctx = Context(h, W, False)
    ctx.set_walkers(np.concatenate([p.reshape(W, -1) for p in psi], axis=1))
    fb, ov = ctx.force_bias(), ctx.overlaps()
    ctx.close()
    S = [np.einsum("mi,wmj->wij", p, x) for p, x in zip(phi, psi)]
    want = np.linalg.det(S[0]) * np.linalg.det(S[1])
    assert np.max(np.abs(ov - want) / np.abs(want)) <= 1e-11
    ref, top = 0.0, 0.0
    for p, x, s in zip(phi, psi, S):
        th = x @ np.linalg.inv(s)
        R = np.einsum("mi,gmk->gki", p, L)
        ref = ref + np.einsum("gki,wki->wg", R, th)
        top = top + np.einsum("gki,wki->wg", np.abs(R), np.abs(th))
    assert np.all(np.abs(fb - ref) <= 1e-11 * top)
