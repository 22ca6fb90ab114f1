"""Shadow rays of the bounce before the tail, traced by the tail (small frames)
or in a launch of their own (large ones, counted ones): every path's radiance
equals the megakernel's bit for bit on both sides of the rule, whatever bounce
the tail starts at, for paths that end at that bounce with a shadow ray still to
trace, with one frame in flight and two, and through a captured graph."""
import numpy as np
import pytest

from kittlespt_amd import abi, scenes
from kittlespt_amd.context import Context
from common import settings, view_proj

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    sc = scenes.scene_plain(subdiv=3)
    c.upload(sc)
    yield sc, c
    c.close()


def image(sc, ctx, W, H, integrator, depth, spp, counting=False, **knobs):
    ctx.set_settings(settings(max_depth=depth, integrator=integrator, sun_theta=sc.sun_theta))
    ctx.resize(W, H)
    ctx.set_view(*view_proj(sc, W, H))
    ctx.set_tuning(**{**dict(tail=1, overlap=1, graph=0, ray_sort=0), **knobs})
    ctx.set_trace_counting(counting)
    ctx.render(spp)
    ctx.set_trace_counting(False)
    return ctx.readback(1).view(np.uint32)


# 2^19 pixels is 1024 x 512, 2^21 is 2048 x 1024: at and just above each
@pytest.mark.parametrize("W,H,spp", ((8, 8, 1), (67, 45, 3), (1024, 512, 2), (1024, 513, 2), (2048, 1024, 1),
                                     (2048, 1025, 1)))
@pytest.mark.parametrize("depth", (1, 4))
def test_equals_the_megakernel(ctx, W, H, spp, depth):
    sc, c = ctx
    print(f"[shadow tail] {W}x{H}, {spp} spp, depth {depth}", flush=True)
    want = image(sc, c, W, H, abi.INTEGRATOR_MEGAKERNEL, depth, spp)
    got = image(sc, c, W, H, abi.INTEGRATOR_WAVEFRONT, depth, spp)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("knobs", (dict(tail=0), dict(tail=2), dict(tail=3), dict(overlap=0), dict(graph=1),
                                   dict(ray_sort=1), dict(suspend=64), dict(suspend=0, stack=8, block=64),
                                   dict(counting=True)))
def test_knobs(ctx, knobs):
    sc, c = ctx
    print(f"[shadow tail] 160x90, 4 spp, {knobs}", flush=True)
    want = image(sc, c, 160, 90, abi.INTEGRATOR_MEGAKERNEL, 6, 4)
    keep = c.tuning()
    try:
        got = image(sc, c, 160, 90, abi.INTEGRATOR_WAVEFRONT, 6, 4, **knobs)
    finally:
        c.set_tuning(**keep)
    assert np.array_equal(got, want)


@pytest.fixture(scope="module")
def instanced():
    c = Context(0)
    sc = scenes.scene_instanced_small()
    c.upload(sc)
    yield sc, c
    c.close()


@pytest.mark.parametrize("W,H,spp", ((67, 45, 1), (67, 45, 3), (1024, 512, 2), (1024, 513, 2), (2048, 1024, 1),
                                     (2048, 1025, 1)))
@pytest.mark.parametrize("tail", (1, 2))
def test_instances_equal_the_megakernel(instanced, W, H, spp, tail):
    sc, c = instanced
    print(f"[shadow tail] instances, {W}x{H}, {spp} spp, tail {tail}", flush=True)
    want = image(sc, c, W, H, abi.INTEGRATOR_MEGAKERNEL, 4, spp)
    got = image(sc, c, W, H, abi.INTEGRATOR_WAVEFRONT, 4, spp, tail=tail)
    assert np.array_equal(got, want)


# the rule goes by the batch's pixels: 3 x 64 x 48, and 2^21 of them and 2048 more
@pytest.mark.parametrize("sizes", (((64, 48), (37, 29), (1, 1)), ((1024, 1024), (512, 2048)),
                                   ((1024, 1024), (512, 2048), (64, 32))))
@pytest.mark.parametrize("tail", (1, 2))
def test_view_batches(instanced, sizes, tail):
    sc, c = instanced
    eye, to = np.array(sc.camera_eye, np.float64), np.array(sc.camera_target, np.float64)
    views = [(scenes.perspective_fov_lh(sc.camera_fov, w, h, 1.0, 100.0),
              scenes.look_at_view(eye * (1 + 0.1 * k), to), w, h) for k, (w, h) in enumerate(sizes)]
    c.set_settings(settings(max_depth=5, integrator=abi.INTEGRATOR_WAVEFRONT, sun_theta=sc.sun_theta))
    keep = c.tuning()
    try:
        got = {}
        for t in (0, tail):
            print(f"[shadow tail] views {sizes}, tail {t}", flush=True)
            c.set_tuning(tail=t, graph=0, ray_sort=0)
            got[t] = c.render_views(views, spp=2)
    finally:
        c.set_tuning(**keep)
    for a, b in zip(got[0], got[tail]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
