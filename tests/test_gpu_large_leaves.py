"""Leaves of 64 and more triangles, which the whole wave tests together: sizes
round the wave's 64 and its multiples, ties between equal distances within a
leaf and between instances, closest and any hit, counted and not; bit-exact
against the oracle.  And their cost: a triangle of a large leaf costs no more
than one of a small leaf."""
import ctypes as C
import time

import numpy as np
import pytest

import oracle
from kittlespt_amd import abi, scenes
from kittlespt_amd.context import Context, DeviceBuffer

pytestmark = pytest.mark.gpu

SIZES = (63, 64, 65, 127, 128, 129, 200, 1030)
BASE = np.array([[-2.0, -2.0, 0.0], [2.0, -2.0, 0.0], [0.0, 4.0, 0.0]])


def star(n, seed, width=1.0):
    """n triangles whose centroids are exactly the origin, so that no plane
    splits them: one leaf.  Few distinct scales, so that many are equal."""
    rng = np.random.default_rng(seed)
    p = BASE * rng.choice([0.125, 0.1875, 0.25], n)[:, None, None]
    p[:, :, 0] *= width
    turn = np.array([[0, 1, 2], [2, 0, 1], [1, 2, 0]])[rng.integers(0, 3, n)]
    p = np.take_along_axis(p, turn[:, None, :].repeat(3, 1), 2)
    nr = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
    nr /= np.linalg.norm(nr, axis=1, keepdims=True)
    return p, np.repeat(nr[:, None], 3, 1), rng.random((n, 3, 2)), np.zeros(n, np.int32)


def star_scene(sizes, width=1.0):
    """One mesh per size; three instances of each: two in the same place (ties
    between instances) and one turned."""
    rng = np.random.default_rng(9)
    k = len(sizes)
    at = [scenes.trs(translate=(2.5 * m, 0, 0)) for m in range(k)]
    turned = [scenes.trs(translate=(2.5 * m, 2.5, 0), rotate=scenes.random_rotation(rng)) for m in range(k)]
    return scenes._pack([star(n, n, width) for n in sizes], [scenes.material()], None,
                        instance_mesh=np.tile(np.arange(k, dtype=np.int32), 3),
                        instance_model=np.stack(at + at + turned))


def star_rays(n, count, seed):
    rng = np.random.default_rng(seed)
    rays = np.zeros(n, abi.RAY_DTYPE)
    target = np.stack([2.5 * rng.integers(0, count, n), 2.5 * rng.integers(0, 2, n), np.zeros(n)], 1)
    target = target + rng.uniform(-0.6, 0.6, (n, 3))
    d = rng.normal(size=(n, 3))
    d[rng.random(n) < 0.25, :2] = 0.0          # axis-parallel: zero components, infinite reciprocals
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    rays["org"], rays["dir"] = target - 3.0 * d, d
    rays["tmax"] = np.where(rng.random(n) < 0.3, rng.uniform(2.0, 4.0, n), np.inf)
    return rays


@pytest.fixture(scope="module")
def ctxs():
    sc = star_scene(SIZES)
    ctx = Context(0)
    ctx.upload(sc)
    orc = oracle.OracleScene(sc)
    yield ctx, orc
    ctx.close()
    orc.close()


@pytest.mark.parametrize("n", (1, 63, 64, 65, 20_000))
def test_large_leaves_equal_the_oracle(ctxs, n):
    ctx, orc = ctxs
    for mesh, size in enumerate(SIZES):
        assert list(ctx.blas(mesh)[0]["count"]) == [size]      # one leaf
    rays = star_rays(n, len(SIZES), n)
    print(f"[large leaves] {n} rays", flush=True)
    o, _, _ = orc.trace(rays, oracle.MODE_CLOSEST)
    _, bounded, _ = orc.trace(rays, oracle.MODE_CLOSEST_ENTRY_BOUND)
    g = ctx.trace_closest(rays)
    gc, counts = ctx.trace_closest(rays, counted=True)
    for got in (g, gc):
        assert np.array_equal(got["prim_id"], o["prim_id"]) and np.array_equal(got["inst_id"], o["inst_id"])
        hit = o["prim_id"] >= 0
        assert np.array_equal(got["t"][hit].view(np.uint32), o["t"][hit].view(np.uint32))
        assert np.array_equal(got["bary"][hit].view(np.uint32), o["bary"][hit].view(np.uint32))
        assert np.all(np.isinf(got["t"][~hit]))
    for key in ("tri_tests", "blas_leaf_pops", "blas_entries"):
        assert counts[key] == bounded[key], key
    if n > 1000:
        assert hit.mean() > 0.3 and counts["tri_tests"] > 100 * n
    assert np.array_equal(ctx.trace_any(rays), orc.trace(rays, oracle.MODE_ANY)[0])


def test_large_leaves_in_frames(ctxs):
    """The path tracer's kernels, whose waves mix closest-hit and shadow rays."""
    from common import settings, view_proj
    ctx, orc = ctxs
    sc = ctx.scene
    sc.camera_eye, sc.camera_target = (8.0, 5.0, -9.0), (8.0, 1.0, 0.0)
    W, H = 70, 41
    pix = np.arange(W * H, dtype=np.int32)
    for integrator in (abi.INTEGRATOR_MEGAKERNEL, abi.INTEGRATOR_WAVEFRONT):
        st = settings(max_depth=4, integrator=integrator, sun_theta=sc.sun_theta)
        ctx.set_settings(st)
        ctx.resize(W, H)
        ctx.set_view(*view_proj(sc, W, H))
        cam = ctx.camera()
        print(f"[large leaves] {W}x{H}, integrator {integrator}", flush=True)
        ctx.render(1)
        want = orc.render_pixels(st, cam, W, H, pix, 0, 1)
        assert np.array_equal(ctx.estimate().reshape(-1, 3).view(np.uint32), want.view(np.uint32))


def _us_per_test(size, n, seed):
    """Microseconds per triangle test of n rays among 216 turned instances of
    one leaf of `size` narrow triangles, the best of six launches."""
    rng = np.random.default_rng(seed)
    grid = np.stack(np.meshgrid(*[np.arange(6)] * 3), -1).reshape(-1, 3) * 10.0 + rng.uniform(-2, 2, (216, 3))
    sc = scenes._pack([star(size, size, 0.03125)], [scenes.material()], None, instance_mesh=np.zeros(216, np.int32),
                      instance_model=np.stack([scenes.trs(translate=g, rotate=scenes.random_rotation(rng), scale=4.0)
                                               for g in grid]))
    ctx = Context(0)
    try:
        ctx.upload(sc)
        rays = np.zeros(n, abi.RAY_DTYPE)
        d = rng.normal(size=(n, 3))
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        rays["org"], rays["dir"], rays["tmax"] = rng.uniform(0, 50, (n, 3)), d, np.inf
        dr, dh = DeviceBuffer.from_array(rays), DeviceBuffer(n * abi.HIT_DTYPE.itemsize)
        cnt = abi.KptTraceCounters()
        abi.check(ctx.h, ctx.L.kpt_trace_closest_counted(ctx.h, dr.ptr, dh.ptr, n, C.byref(cnt)))
        tests = cnt.as_dict()["tri_tests"]
        best = float("inf")
        for _ in range(6):
            t = time.perf_counter()
            abi.check(ctx.h, ctx.L.kpt_trace_closest(ctx.h, dr.ptr, dh.ptr, n))
            abi.check(ctx.h, ctx.L.kpt_sync(ctx.h))
            best = min(best, time.perf_counter() - t)
        print(f"[large leaves] leaf of {size}: {tests} tests, {best * 1e6:.0f} us", flush=True)
        return best * 1e6 / tests
    finally:
        ctx.close()


def test_a_large_leafs_triangle_costs_no_more_than_a_small_leafs():
    """Over 10^8 and more tests each, so that a launch is milliseconds.  Measured:
    0.76 of the small leaf's cost; 1.9 with each lane at its own large leaf."""
    small = _us_per_test(63, 1 << 20, 4)
    large = _us_per_test(4096, 1 << 17, 4)
    print(f"[large leaves] {small * 1e6:.2f} ps a test in leaves of 63, {large * 1e6:.2f} in leaves of 4096", flush=True)
    assert large <= 1.25 * small
