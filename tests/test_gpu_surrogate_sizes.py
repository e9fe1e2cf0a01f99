"""Training kernels of the surrogate at the sizes where their tiles end: blocks of 32 rows, staged
chunks of 256, bias sums of 256 rows a turn."""
import numpy as np
import pytest

import mlp_oracle as M
import pimc_hip as ph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 255, 257, 512, 513, 769, 2049])
def test_gradient_at_the_edges_of_tiles(n):
    """Against FP64.  Operands rounded to BF16 (2^-9) pass through at most eight products on the way
    to a weight's gradient: 8 * 2^-9 = 1.6e-2 of each block's norm, with targets far from the outputs
    so that dL/dout does not cancel; the loss takes the four of the way forward, twice (a square)."""
    rng = np.random.default_rng(n)
    theta = (M.glorot(2) + rng.normal(0, 0.02, M.NW)).astype(np.float32)
    X = rng.normal(0, 1, (n, 4)).astype(np.float32)
    y = rng.normal(4, 1, n).astype(np.float32)
    ctx = ph.Context(1, seed=3)
    loss, g = ctx.surrogate_grad(theta, X, y)
    again = ctx.surrogate_grad(theta, X, y)
    ctx.close()
    lo, go = M.loss_grad(theta.astype(np.float64), X, y)
    assert abs(loss - lo) <= 1.6e-2 * lo
    for k, (o, s) in M.OFF.items():
        m = int(np.prod(s))
        assert np.linalg.norm(g[o:o + m] - go[o:o + m]) <= 1.6e-2 * np.linalg.norm(go[o:o + m]), k
    assert loss == again[0] and np.array_equal(g, again[1])


def test_a_step_is_adam_on_the_gradient():
    """One epoch of one batch: Adam's first step moves every weight by lr times the gradient's sign,
    so what training returns minus its start is that of the gradient at its own start."""
    rng = np.random.default_rng(4)
    n, lr = 65, 1e-3
    X = rng.normal(0, 1, (n, 4)).astype(np.float32)
    v = rng.normal(0, 1, n).astype(np.float32)
    ctx = ph.Context(1, seed=3)
    ctx.surrogate_train(X, v, epochs=1, batch=n, lr=1e-30, seed=9)  # a step too small to see: the start
    t0, norm = ctx.surrogate_get()
    ctx.surrogate_train(X, v, epochs=1, batch=n, lr=lr, seed=9)
    t1, _ = ctx.surrogate_get()
    xn, yn = (X - norm[:4]) / norm[4:8], (v - norm[8]) / norm[9]
    _, g = ctx.surrogate_grad(t0, xn, yn)  # the rows in another order: the sums' last bits differ
    ctx.close()
    clear = np.abs(g) > 1e-4  # Adam's 1e-8 beside |g| then takes at most 1e-4 of the step
    assert clear.sum() > 1000
    step = (t0.astype(np.float64) - t1)[clear]
    # FP32 weights of size < 1 hold a step to 2^-24
    assert np.abs(step - lr * np.sign(g[clear])).max() <= 2.0 ** -23 + 1e-4 * lr
