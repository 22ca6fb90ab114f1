"""The training records of a frame, wherever their paths' vertices and shadow
rays run: in the stage kernels, in the path-per-lane tail, or in the tail with
the shadow ray of the bounce before it (small frames).  A record's target is
the radiance its path gathered past the cache vertex, so it needs the radiance
so far at that vertex exactly, with the vertex's own estimate or without.

Every path trains (train_samples at least the frame's pixels) in one step, so
the step's gradient and loss are sums over all records: compared with the
oracle's over its own records, and between the routes.  One record of n that is
missing or has another target moves them by about 1/n, at least 2^-13 at these
sizes.  Tolerance: the sums are FP32, of the same terms in the order of the
paths' arrival (two runs of one route differ by 2e-7), and against the oracle a
layer's sum on a rounding boundary can give the neighbouring BF16 activation,
2^-8 of one of 64, in few of the n samples."""
import numpy as np
import pytest

import oracle
from kittlespt_amd import abi, scenes
from kittlespt_amd.context import Context
from common import settings, view_proj
from test_cache_oracle import he_weights

pytestmark = pytest.mark.gpu

BOXES = {"plain": ((-20.0, -1.0, -20.0), (20.0, 3.0, 20.0)), "instanced": ((0.0, 0.0, 0.0), (100.0, 100.0, 100.0))}
SCALE = 1e4
WEIGHTS = he_weights(41) * np.float32(0.5)


@pytest.fixture(scope="module", params=("plain", "instanced"))
def scene(request):
    sc = scenes.scene_plain(subdiv=3) if request.param == "plain" else scenes.scene_instanced_small()
    if request.param == "instanced":     # from near one instance: more paths reach their cache vertex
        m = sc.instance_model[18].reshape(4, 4)
        size = np.linalg.norm(m[0, :3])
        sc.camera_target = tuple(m[3, :3])
        sc.camera_eye = tuple(m[3, :3] + size * np.array([0.36, 0.96, -1.92]))
    ctx = Context(0)
    ctx.upload(sc)
    yield request.param, sc, ctx
    ctx.close()


def trained(which, sc, ctx, W, H, depth, *, tail, frames=1, enabled=False, nee=0, wide=0.0, rate=1e-3,
            **knobs):
    """Gradient, loss, records and image of `frames` frames in which every path trains."""
    keep = ctx.tuning()
    try:
        ctx.set_tuning(**{**dict(tail=tail, overlap=1, graph=0, ray_sort=0), **knobs})
        ctx.set_settings(settings(max_depth=depth, integrator=abi.INTEGRATOR_WAVEFRONT, sun_theta=sc.sun_theta))
        ctx.resize(W, H)
        ctx.set_view(*view_proj(sc, W, H))
        ctx.cache_configure(enabled=enabled, train=True, train_samples=W * H, train_steps=1, seed=7,
                            bounds=BOXES[which], radiance_scale=SCALE, nee_at_vertex=nee, wide_roughness=wide,
                            learning_rate=rate)
        ctx.cache_set_weights(WEIGHTS)
        print(f"[records] {which} {W}x{H}, depth {depth}, tail {tail}, {frames} frames, enabled {enabled}, nee {nee}, "
              f"wide {wide}, {knobs}", flush=True)
        ctx.render(frames)
        s = ctx.cache_stats()
        return ctx.cache_gradient().astype(np.float64), s["loss"], int(s["train_records"]), ctx.readback(1)
    finally:
        ctx.cache_configure(enabled=False, train=False)
        ctx.set_tuning(**keep)


def same(got, want, tol):
    g, loss, n, _ = got
    gw, lw, nw, _ = want
    assert n == nw and n > 0
    assert np.linalg.norm(g - gw) <= tol * np.linalg.norm(gw)
    assert abs(loss - lw) <= tol * abs(lw)


@pytest.mark.parametrize("tail", (0, 1, 2, 3))
@pytest.mark.parametrize("W,H,depth", ((33, 21, 4), (64, 48, 6)))
def test_records_equal_the_oracles(scene, W, H, depth, tail):
    """Without the vertex's own estimate: the target is the path's whole
    radiance less what came before the vertex, both of which the oracle gives."""
    which, sc, ctx = scene
    got = trained(which, sc, ctx, W, H, depth, tail=tail)
    cam = ctx.camera()
    st = settings(max_depth=depth, integrator=abi.INTEGRATOR_WAVEFRONT, sun_theta=sc.sun_theta)
    orc = oracle.OracleScene(sc)
    try:
        before, q = orc.render_cache_queries(st, cam, W, H, 0)
        end = orc.render_pixels(st, cam, W, H, np.arange(W * H, dtype=np.int32), 0, 1)
    finally:
        orc.close()
    hit = q[:, 0] > 0
    assert np.abs(end).max() < 1e8                      # no radiance at the output's clamp
    bq = q[hit, 8:11]
    with np.errstate(divide="ignore", invalid="ignore"):
        suffix = np.where(bq > 0, ((end[hit] - before[hit]) / bq) / np.float32(SCALE), np.float32(0))
    n = int(hit.sum())
    target = np.concatenate([suffix, np.zeros((n, 1))], 1).astype(np.float32)
    dirs = np.concatenate([q[hit, 5:8], np.zeros((n, 1))], 1).astype(np.float32)
    loss, g = oracle.cache_loss_grad(WEIGHTS, q[hit, 1:5], dirs, target, *BOXES[which], mode=0)
    same(got, (np.asarray(g, np.float64), loss, n, None), 1e-5)


@pytest.mark.parametrize("enabled,wide", ((False, 0.0), (True, 0.0), (True, 0.7), (False, 0.7)))
@pytest.mark.parametrize("nee", (0, 1))
@pytest.mark.parametrize("tail", (1, 2, 3))
def test_routes_make_the_same_records(scene, tail, nee, enabled, wide):
    """Against the stage kernels (tail 0): records, gradient and, of the first
    frame, the image bit for bit."""
    which, sc, ctx = scene
    for W, H in ((33, 21), (120, 67)):
        kw = dict(enabled=enabled, nee=nee, wide=wide)
        want = trained(which, sc, ctx, W, H, 6, tail=0, **kw)
        got = trained(which, sc, ctx, W, H, 6, tail=tail, **kw)
        same(got, want, 2e-6)
        if not enabled:
            assert np.array_equal(got[3].view(np.uint32), want[3].view(np.uint32))


@pytest.mark.parametrize("knobs", (dict(graph=1), dict(ray_sort=1), dict(suspend=0), dict(suspend=64),
                                   dict(stack=8, block=64), dict(sort=1), dict(overlap=0)))
def test_knobs(scene, knobs):
    which, sc, ctx = scene
    kw = dict(nee=1, enabled=True, wide=0.7)
    same(trained(which, sc, ctx, 120, 67, 6, tail=1, **kw, **knobs), trained(which, sc, ctx, 120, 67, 6, tail=0, **kw),
         2e-6)


# one frame: 2^21 pixels (2048 x 1024) and just above; two in flight: 2^18 (512 x 512)
# and just below, 2^19 (1024 x 512) and just above.  With a learning rate that
# moves no weight, the second frame's gradient is of the same network.
@pytest.mark.parametrize("W,H,frames", ((2048, 1024, 1), (2048, 1025, 1), (512, 512, 2), (512, 511, 2), (1024, 512, 2),
                                        (1024, 513, 2), (120, 67, 3)))
@pytest.mark.parametrize("tail", (1, 2))
def test_both_sides_of_the_rule(scene, W, H, frames, tail):
    which, sc, ctx = scene
    kw = dict(nee=1, frames=frames, rate=1e-30)
    want = trained(which, sc, ctx, W, H, 4, tail=0, overlap=0, **kw)
    got = trained(which, sc, ctx, W, H, 4, tail=tail, **kw)
    same(got, want, 2e-6)
    assert np.array_equal(got[3].view(np.uint32), want[3].view(np.uint32))
