"""The cache network at the sizes where its kernels' tiles end: 16 queries or
samples per tile, 64 samples per training workgroup, 16 partial sums per Adam
workgroup; against the oracle's BF16-rounding forward and backward.

Tolerance: sums differ in order only, below 1e-6 of the result, but one within
that of a BF16 rounding boundary gives the neighbouring activation, 2^-8 of its
value away, and moves its query's outputs by up to 2^-8 of their scale and its
sample's gradient by up to 2^-8 of its size.  Few queries have such a sum (5 of
4097 measured; the others equal the oracle's to the last bit or two), and with
the backward pass's sums about one sample in 64."""
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
    off = np.abs(got - want).max(1) / np.abs(want).max()
    print(f"[cache] forward: {int((off > 1e-6).sum())} of {n} queries off, most {off.max():.1e}", flush=True)
    assert off.max() <= 2.0 ** -8 and (off > 1e-6).sum() <= 1 + n / 256


def samples(w, n):
    """n training samples whose outputs are not near zero, where the relative
    loss magnifies the last bit of an activation."""
    pos, dirs = queries(32 * n + 64, n + 1)
    keep = np.abs(oracle.cache_forward(w, pos, dirs, BMIN, BMAX, mode=0)[:, :3]).min(1) > 0.5
    t = np.zeros((n, 4), np.float32)
    t[:, :3] = np.random.default_rng(n).uniform(0, 2, (n, 3))
    pos, dirs = pos[keep][:n], dirs[keep][:n]
    assert len(pos) == n
    return pos, dirs, t


@pytest.mark.parametrize("n,steps", ((1, 1), (16, 1), (63, 1), (64, 1), (65, 1), (130, 3), (1030, 1), (1030, 16),
                                     (10, 7), (65, 16)))
def test_training_step(ctx, n, steps):
    """The gradient and loss of the last step that had samples, of `steps` over
    n samples (batches of ceil(n / steps), the last one ragged; the last two of
    (10, 7) and three of (65, 16) empty), and the weights after them all."""
    w = he_weights(22)
    ctx.cache_set_weights(w)
    pos, dirs, t = samples(w, n)
    print(f"[cache] {steps} training steps over {n} samples", flush=True)
    loss = ctx.cache_train(pos, dirs, t, steps=steps)
    got = ctx.cache_gradient().astype(np.float64)
    batch = -(-n // steps)
    m, v = np.zeros_like(w), np.zeros_like(w)
    for k in range(steps):
        sl = slice(k * batch, min(n, (k + 1) * batch))
        if sl.start >= n:
            break
        before, b = w, sl.stop - sl.start
        lo, g = oracle.cache_loss_grad(w, pos[sl], dirs[sl], t[sl], BMIN, BMAX, mode=0)
        w, m, v = oracle.cache_adam(w, m, v, np.asarray(g, np.float32), k + 1, 1e-3)
    off = np.linalg.norm(got - g) / np.linalg.norm(g)
    woff = np.linalg.norm(ctx.cache_weights() - w) / np.linalg.norm(w - he_weights(22))
    lost = 1.0
    if b > 1:
        cut = slice(sl.start, sl.stop - 1)
        gl = oracle.cache_loss_grad(before, pos[cut], dirs[cut], t[cut], BMIN, BMAX, mode=0)[1]
        lost = np.linalg.norm(np.asarray(gl) * (b - 1) / b - g) / np.linalg.norm(g)
    print(f"[cache] loss off {abs(loss / lo - 1):.1e}, gradient {off:.1e} (a sample lost {lost:.1e}), weights {woff:.1e}", flush=True)
    tol = 2.0 ** -8 * max(1 / b, 1 / 64)
    assert lost > 20 * tol
    assert off <= tol
    assert loss == pytest.approx(lo, rel=1e-5)
    # of all the steps' movement, of which one step more or less is a thirteenth
    # at least (a gradient near zero can take the other sign in Adam's first step)
    assert woff <= 1e-2
