"""The surrogate's gradients over batches at the edges of the chunks the weight gradients are
summed in (128 rows at least), against the numpy oracle.

Both sides round the same GEMM operands to bf16; they differ where FP32 accumulation moves an
operand across a rounding boundary (a 2^-8 change of a few operands in 10^4) and by the FP32
sums over the batch: 1e-2 of a gradient's norm is well above both."""
import os
import sys

import numpy as np
import pytest

from test_gpu_parity import build

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,hidden", [(1, 16), (63, 64), (255, 64), (256, 65), (385, 64), (1000, 130), (4096, 64)])
def test_gradients_of_batch(rows, hidden):
    h, _, ctx, _ = build("c1_small", 8)
    ctx.surrogate_init(hidden=hidden, seed=3)
    F = h.nchol + 2 * h.norb
    dims = [F, hidden, hidden, hidden, 1]
    rng = np.random.default_rng(rows)
    p = ctx.surrogate_params()
    nw = sum(dims[i] * dims[i + 1] + dims[i + 1] for i in range(4))
    p[nw:nw + F] = rng.normal(0, 0.1, F)
    p[nw + F:nw + 2 * F] = rng.uniform(0.5, 2.0, F)
    p[-2], p[-1] = 0.3, 2.0
    ctx.surrogate_params(p)
    X = rng.standard_normal((rows, F)).astype(np.float32)
    t = (X[:, :5].sum(axis=1) + rng.normal(0.0, 1.0, rows)).astype(np.float32)
    loss, g = ctx.surrogate_grad(X, t)
    ctx.close()
    loss_o, go = mlp_oracle.loss_and_grads(p, dims, X, t)
    assert abs(loss - loss_o) <= 1e-3 * abs(loss_o)
    off = 0
    for i in range(4):
        for n in (dims[i] * dims[i + 1], dims[i + 1]):
            a, b = g[off:off + n], go[off:off + n]
            assert np.linalg.norm(a - b) <= 1e-2 * np.linalg.norm(b) + 1e-7, (i, n)
            off += n
