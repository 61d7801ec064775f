"""Results that reach the host through pinned memory and those too large for it, and the kept
workspace of ham_and_overlap: grown, given back past its bound, and shared by threads."""
import threading

import numpy as np
import pytest

from vmc_amd.abi import HamArrays
from vmc_amd.afqmc import Context

pytestmark = pytest.mark.gpu


def system(N, n, G, seed):
    rng = np.random.default_rng(seed)
    L = rng.standard_normal((G, N, N)) / N
    L = L + np.swapaxes(L, 1, 2)
    h1 = rng.standard_normal((N, N))
    phi = [np.linalg.qr(rng.standard_normal((N, n)))[0] for _ in range(2)]
    return HamArrays(N, n, n, 0.5, h1 + h1.T, h1 + h1.T, L, phi[0], phi[1]), rng


@pytest.mark.parametrize("W", [1, 6553, 6554, 32768, 32769])   # (energy, <H>, overlap): 5 W words, the weights W
def test_sizes_round_trip(W):
    h, rng = system(2, 1, 1, W)
    ctx = Context(h, W, False)
    over = rng.uniform(0.5, 2.0, W) + 0j
    weights = rng.uniform(0.5, 2.0, W)
    dets = np.array([h.serial_det(h.phi_up, h.phi_dn)]) * rng.uniform(0.5, 2.0, (W, 1))
    ctx.set_walkers(dets, overlaps=over, weights=weights)
    e, ho = ctx.measure()
    got = ctx.get_walkers()
    assert np.array_equal(ctx.weights(), weights) and np.array_equal(got[2], weights)
    assert np.array_equal(got[0], dets) and np.max(np.abs(got[1] - over)) <= 1e-14 * 2.0
    # <H> / overlap is the local energy (walker for walker), the same for every multiple of one determinant
    ho = ho.reshape(W, -1)
    assert np.max(np.abs((ho[:, 0] / ho[:, 1]).real - e)) <= 1e-13 * np.max(np.abs(e)) + 1e-13
    assert np.max(np.abs(e - e[0])) <= 1e-12 * max(1.0, abs(e[0]))
    ctx.close()


def test_workspace_grows_is_given_back_and_shared():
    h, rng = system(64, 60, 4, 1)
    ctx = Context(h, 2, False)
    base = [h.serial_det(*(p + 0.05 * (rng.standard_normal(p.shape) + 1j * rng.standard_normal(p.shape))
                           for p in (h.phi_up, h.phi_dn))) for _ in range(7)]
    one = np.array([ctx.ham_and_overlap(d[None, :], h.nchol)[0] for d in base])
    for count in (3, 600, 2, 7):     # 600: past what is kept
        dets = np.array([base[i % 7] for i in range(count)])
        got = ctx.ham_and_overlap(dets, h.nchol)
        want = one[np.arange(count) % 7]
        assert np.max(np.abs(got - want) / np.abs(want)) <= 1e-11
    serial = [ctx.ham_and_overlap(np.array(base[:k]), h.nchol) for k in range(1, 8)]
    out = [None] * 7

    def work(k):
        for _ in range(5):
            out[k] = ctx.ham_and_overlap(np.array(base[:k + 1]), h.nchol)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(7)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    ctx.close()
    assert all(np.array_equal(a, b) for a, b in zip(out, serial))
