"""The cache network at the sizes where its kernels' tiles end: 16 queries or
samples per tile, 64 samples per training workgroup, 16 partial sums per Adam
workgroup; against the oracle's BF16-rounding forward and backward.

Tolerance: sums differ in order only, but a sum on a rounding boundary can give
the neighbouring BF16 activation, 2^-8 of its value away, of the 64 or more
that reach each output: below 2^-8 of the outputs' scale in an output and of
the gradient's norm."""
import numpy as np
import pytest

import oracle
from kittlespt_amd.context import Context
from test_cache_oracle import BMAX, BMIN, he_weights, queries

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    c.cache_configure(bounds=(BMIN, BMAX), seed=3)
    yield c
    c.close()


@pytest.mark.parametrize("n", (1, 15, 16, 17, 63, 64, 65, 4097))
def test_forward(ctx, n):
    w = he_weights(21)
    ctx.cache_set_weights(w)
    pos, dirs = queries(n, n)
    print(f"[cache] forward {n} queries", flush=True)
    got = ctx.cache_infer(pos, dirs)[:, :3].astype(np.float64)
    want = oracle.cache_forward(w, pos, dirs, BMIN, BMAX, mode=0)
    assert np.abs(got - want).max() <= 2.0 ** -8 * np.abs(want).max()


@pytest.mark.parametrize("n,steps", ((1, 1), (16, 1), (63, 1), (64, 1), (65, 1), (130, 3), (1030, 1), (1030, 16)))
def test_training_step(ctx, n, steps):
    """The gradient of the last step of `steps` over n samples (batches of
    ceil(n / steps), the last one ragged or empty)."""
    w = he_weights(22)
    ctx.cache_set_weights(w)
    pos, dirs = queries(n, n + 1)
    t = np.zeros((n, 4), np.float32)
    t[:, :3] = np.random.default_rng(n).uniform(0, 2, (n, 3))
    print(f"[cache] {steps} training steps over {n} samples", flush=True)
    loss = ctx.cache_train(pos, dirs, t, steps=steps)
    got = ctx.cache_gradient().astype(np.float64)
    batch = -(-n // steps)
    m, v = np.zeros_like(w), np.zeros_like(w)
    for k in range(steps):
        sl = slice(k * batch, min(n, (k + 1) * batch))
        if sl.start >= n:
            break
        lo, g = oracle.cache_loss_grad(w, pos[sl], dirs[sl], t[sl], BMIN, BMAX, mode=0)
        w, m, v = oracle.cache_adam(w, m, v, np.asarray(g, np.float32), k + 1, 1e-3)
    assert loss == pytest.approx(lo, rel=2.0 ** -8)
    assert np.linalg.norm(got - g) <= 2.0 ** -8 * np.linalg.norm(g)
