"""The weight gradients' chain of products takes its rows in chunks of 24 groups of 16, staged two
ahead: batches that end a chunk, begin the next, and fill one, two and three."""
import numpy as np
import pytest

import mlp_oracle as M
import pimc_hip as ph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [368, 384, 385, 767, 768, 800, 1152, 1153])
def test_gradient_at_the_edges_of_chunks(n):
    """Against FP64, with the bound of eight products of BF16 operands: 8 * 2^-9 of each block's norm."""
    rng = np.random.default_rng(n)
    theta = (M.glorot(2) + rng.normal(0, 0.02, M.NW)).astype(np.float32)
    X = rng.normal(0, 1, (n, 4)).astype(np.float32)
    y = rng.normal(4, 1, n).astype(np.float32)
    ctx = ph.Context(1, seed=3)
    loss, g = ctx.surrogate_grad(theta, X, y)
    ctx.close()
    lo, go = M.loss_grad(theta.astype(np.float64), X, y)
    assert abs(loss - lo) <= 1.6e-2 * lo
    for k, (o, s) in M.OFF.items():
        m = int(np.prod(s))
        assert np.linalg.norm(g[o:o + m] - go[o:o + m]) <= 1.6e-2 * np.linalg.norm(go[o:o + m]), k
