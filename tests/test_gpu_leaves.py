"""Leaves whose triangles are spread over a wave's lanes: every leaf size at
which the split changes (one triangle, a wave's 64, larger leaves than an
entry holds), ray counts around a wave and a workgroup, ties between equal
distances, and rays at the edges of their interval.  Bit-exact against the
oracle, as the traversal's contract is (no tolerance)."""
import numpy as np
import pytest

import oracle
from kittlespt_amd import abi, scenes
from kittlespt_amd.context import Context

pytestmark = pytest.mark.gpu

LEAVES = (1, 2, 3, 7, 8, 9, 21, 32, 33, 63, 64, 65, 130)


def leaf_scene():
    """One mesh per leaf size: that many copies of one triangle (no plane
    splits equal centroids, so they share a leaf), every third one shifted along
    the normal; two instances of each, the second coplanar with the first."""
    rng = np.random.default_rng(3)
    meshes = []
    for n in LEAVES:
        p = np.repeat(np.array([[[-0.5, -0.5, 0], [0.5, -0.5, 0], [0, 0.5, 0]]]), n, 0)
        p[2::3, :, 2] += 0.125
        nr = np.tile(np.array([0, 0, 1.0]), (n, 3, 1))
        meshes.append((p, nr, rng.random((n, 3, 2)), np.zeros(n, np.int32)))
    k = len(LEAVES)
    models = []
    for r in range(2):
        for m in range(k):
            models.append(scenes.trs(translate=(1.5 * m, 0, 0), scale=1.0 if r == 0 else 0.75))
    return scenes._pack(meshes, [scenes.material()], None, instance_mesh=np.tile(np.arange(k, dtype=np.int32), 2),
                        instance_model=np.stack(models))


@pytest.fixture(scope="module")
def ctxs():
    sc = leaf_scene()
    ctx = Context(0)
    ctx.upload(sc)
    orc = oracle.OracleScene(sc)
    yield ctx, orc
    ctx.close()
    orc.close()


def leaf_rays(n, seed):
    rng = np.random.default_rng(seed)
    rays = np.zeros(n, abi.RAY_DTYPE)
    target = np.stack([1.5 * rng.integers(0, len(LEAVES), n) + rng.uniform(-0.4, 0.4, n), rng.uniform(-0.4, 0.3, n),
                       np.zeros(n)], 1)
    side = np.where(rng.random(n) < 0.5, -1.0, 1.0)
    org = target + np.stack([rng.uniform(-2, 2, n), rng.uniform(-1, 1, n), side * rng.uniform(0.5, 3, n)], 1)
    straight = rng.random(n) < 0.25                     # axis-parallel: zero components, infinite reciprocals
    org[straight, :2] = target[straight, :2]
    rays["org"], rays["dir"] = org, target - org
    rays["tmax"] = np.inf
    return rays


def check(ctx, orc, rays, what):
    print(f"[leaves] {what}: {len(rays)} rays", flush=True)
    o, _, _ = orc.trace(rays, oracle.MODE_CLOSEST)
    for counted in (False, True):
        g = ctx.trace_closest(rays, counted=counted)
        g = g[0] if counted else g
        assert np.array_equal(g["prim_id"], o["prim_id"]) and np.array_equal(g["inst_id"], o["inst_id"])
        hit = o["prim_id"] >= 0
        assert np.array_equal(g["t"][hit].view(np.uint32), o["t"][hit].view(np.uint32))
        assert np.array_equal(g["bary"][hit].view(np.uint32), o["bary"][hit].view(np.uint32))
        assert np.all(np.isinf(g["t"][~hit]))
    oa, _, _ = orc.trace(rays, oracle.MODE_ANY)
    assert np.array_equal(ctx.trace_any(rays), oa)
    return o


@pytest.mark.parametrize("n", (1, 2, 63, 64, 65, 255, 257, 20_000))
def test_leaf_sizes_and_ray_counts(ctxs, n):
    o = check(*ctxs, leaf_rays(n, n), "every leaf size")
    if n > 1000:
        assert (o["prim_id"] >= 0).mean() > 0.5


def test_interval_edges(ctxs):
    """tmax and tmin at, one step below and one step above a hit's distance,
    negative and empty intervals, and directions without a finite reciprocal."""
    ctx, orc = ctxs
    base = leaf_rays(4096, 77)
    t = orc.trace(base, oracle.MODE_CLOSEST)[0]["t"]
    t = np.where(np.isfinite(t), t, np.float32(1.0)).astype(np.float32)
    for tmin, tmax in ((np.float32(0), t), (np.float32(0), np.nextafter(t, np.float32(np.inf))),
                       (np.float32(0), np.nextafter(t, np.float32(0))), (t, np.float32(np.inf)),
                       (np.nextafter(t, np.float32(0)), np.float32(np.inf)), (np.float32(0), np.float32(0)),
                       (np.float32(0), np.float32(-1)), (np.float32(0), np.float32(3.4028235e38)),
                       (np.float32(2), np.float32(1)), (np.float32(0), np.float32(np.nan))):
        rays = base.copy()
        rays["tmin"], rays["tmax"] = tmin, tmax
        check(ctx, orc, rays, "interval edges")
    rays = base.copy()
    rays["dir"][::4] = 0.0
    rays["dir"][1::4, 0] = np.nan
    rays["dir"][2::4, 1] = np.inf
    rays["dir"][3::4] *= np.float32(1e-38)
    check(ctx, orc, rays, "directions")
