"""What a walker gets does not depend on the walkers it is taken with: the FP64 sums over Cholesky vectors
run in an order fixed by the system, so any number of walkers, any place among them and dead neighbours
give the same bits."""
import numpy as np
import pytest

from vmc_amd.abi import HamArrays
from vmc_amd.afqmc import Context

pytestmark = pytest.mark.gpu

CASES = [
    # N, na, nb, G, RHF trial and walkers
    (12, 3, 2, 50, False),      # fewer than four electrons
    (20, 4, 4, 90, False),      # 16 walkers and vectors a tile
    (30, 11, 8, 130, False),    # slots of different size
    (47, 23, 17, 163, False),   # odd; three waves for one spin
    (64, 20, 20, 400, True),
    (60, 40, 33, 70, False),
    (66, 64, 60, 30, False),    # a walker and a vector a tile
]
COUNTS = [1, 5, 40, 300]


def system(N, na, nb, G, rhf, seed=3):
    rng = np.random.default_rng([seed, N])
    L = rng.standard_normal((G, N, N)) / N
    L = L + np.swapaxes(L, 1, 2)
    h1 = rng.standard_normal((N, N))
    h1 = h1 + h1.T
    phi = [np.linalg.qr(rng.standard_normal((N, n)))[0] for n in (na, nb)]
    h = HamArrays(N, na, nb, 0.0, h1, h1, L, phi[0], phi[0] if rhf else phi[1], trial_rhf=rhf)
    dets = []
    for _ in range(COUNTS[-1]):
        up, dn = (p + 0.1 * (rng.standard_normal(p.shape) + 1j * rng.standard_normal(p.shape)) for p in phi)
        dets.append(h.serial_det(up, up if rhf else dn))
    return h, np.array(dets), rng


@pytest.mark.parametrize("case", CASES, ids=lambda c: "N%d_%d_%d_G%d%s" % (c[:4] + ("_rhf" if c[4] else "",)))
def test_exchange_energy_in_any_company(case):
    h, dets, rng = system(*case)
    keep = h.nchol - 1

    def exchange(pick, weights):
        ctx = Context(h, len(pick), case[4])
        ctx.set_nchol_ene(keep)
        ctx.set_walkers(dets[pick], weights=weights)
        ctx.measure()
        ek = np.array(ctx.energy_parts()[1])
        ctx.close()
        return ek

    every = np.arange(COUNTS[-1])
    want = exchange(every, np.ones(len(every)))
    assert np.all(want != 0.0)
    for count in COUNTS[:-1]:
        for first in (0, 7):
            pick = every[first:first + count]
            assert np.array_equal(exchange(pick, np.ones(count)), want[pick])
    weights = rng.integers(0, 2, len(every)).astype(float)
    got = exchange(every, weights)
    assert np.array_equal(got[weights != 0.0], want[weights != 0.0])


@pytest.mark.parametrize("case", CASES + [
    # the force bias' sum over (orbital, electron) pairs: too short to divide; divided, where theta is
    # larger than the overlap matrices; more vectors than an overlap matrix holds
    (7, 2, 2, 20, False), (150, 40, 36, 230, False), (20, 3, 3, 4200, True),
], ids=lambda c: "N%d_%d_%d_G%d%s" % (c[:4] + ("_rhf" if c[4] else "",)))
def test_force_bias_and_energies_in_any_company(case):
    """Force biases between populations; energies and overlaps also between populations and the calls that
    evaluate given determinants."""
    h, dets, rng = system(*case)
    keep = h.nchol - 1

    def walkers(pick, weights=None):
        ctx = Context(h, len(pick), case[4])
        ctx.set_nchol_ene(keep)
        ctx.set_walkers(dets[pick], weights=weights)
        fb, (energies, ho) = ctx.force_bias(), ctx.measure()
        ctx.close()
        return fb, energies, ho

    every = np.arange(COUNTS[-1])
    fb, energies, ho = walkers(every)
    ctx = Context(h, 1, case[4])
    for count in COUNTS:
        for first in (0, 7):
            pick = every[first:first + count]
            if count < COUNTS[-1]:
                got = walkers(pick)
                assert np.array_equal(got[0], fb[pick]) and np.array_equal(got[1], energies[pick])
            assert np.array_equal(ctx.ham_and_overlap(dets[pick], keep).ravel(), np.asarray(ho).reshape(len(every), -1)[pick].ravel())
    ctx.close()
    weights = rng.integers(0, 2, len(every)).astype(float)
    got, live = walkers(every, weights), weights != 0.0
    assert np.array_equal(got[0][live], fb[live]) and np.array_equal(got[1][live], energies[live])
