"""The comb at the edges of its running sum (16 elements read ahead, pairs of them, chunks held in
LDS) against numpy: the sum is the sequential one, so total, weights and the copied walkers are exact."""
import numpy as np
import pytest

from vmc_amd.abi import HamArrays
from vmc_amd.afqmc import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 2047, 2048, 2049, 4100])
def test_comb_is_the_sequential_sum(W):
    rng = np.random.default_rng(W)
    h = HamArrays(3, 1, 1, 0.0, np.eye(3), np.eye(3), rng.standard_normal((2, 3, 3)), np.eye(3)[:, :1], np.eye(3)[:, :1])
    dets = rng.standard_normal((W, h.mat_size)) + 1j * rng.standard_normal((W, h.mat_size))
    weights = rng.uniform(0.0, 2.0, W)
    weights[W // 2] = 0.0 if W > 1 else 1.0
    ctx = Context(h, W, False)
    ctx.set_walkers(dets, overlaps=dets[:, 0].copy(), weights=weights)
    total = ctx.comb(0.3)
    got, over, after = ctx.get_walkers()
    ctx.close()
    cum = np.cumsum(weights)
    pick = np.minimum(np.searchsorted(cum, (np.arange(W) + 0.3) / W * cum[-1]), W - 1)
    assert total == cum[-1]
    assert np.array_equal(after, np.full(W, cum[-1] / W))
    assert np.array_equal(got, dets[pick]) and np.max(np.abs(over - dets[pick, 0])) <= 1e-14 * np.max(np.abs(over))   # kept as a logarithm

