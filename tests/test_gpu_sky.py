"""The sky's density profile evaluated without its divisions and range checks:
frames of an empty scene looking up, along the horizon and straight down (where
the path through the planet leaves the shortened exponential's range), with the
sun below, at and above the horizon, equal the oracle's bit for bit."""
import math

import numpy as np
import pytest

import oracle
from kittlespt_amd import abi, scenes
from kittlespt_amd.context import Context
from common import settings
from test_gpu_edge import _empty

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("integrator", (abi.INTEGRATOR_MEGAKERNEL, abi.INTEGRATOR_WAVEFRONT))
@pytest.mark.parametrize("sun_deg", (-5.0, 0.0, 0.5, 30.0, 90.0))
def test_sky_equals_the_oracle(sun_deg, integrator):
    sc = _empty(False)
    W, H = 40, 25
    ctx, orc = Context(0), oracle.OracleScene(sc)
    try:
        ctx.upload(sc)
        st = settings(max_depth=2, integrator=integrator, sun_theta=math.radians(sun_deg))
        ctx.set_settings(st)
        ctx.resize(W, H)
        for target in ((0.1, 5.0, 0.0), (4.0, 1.2, 1.0), (0.1, -5.0, 0.2)):
            ctx.set_view(scenes.perspective_fov_lh(math.radians(100.0), W, H, 1.0, 100.0),
                         scenes.look_at_view((0.0, 1.2, 0.0), target))
            print(f"[sky] sun {sun_deg} deg, looking at {target}, integrator {integrator}", flush=True)
            cam = ctx.camera()
            ctx.reset()
            ctx.render(1)
            got = ctx.estimate().reshape(-1, 3)
            want = orc.render_pixels(st, cam, W, H, np.arange(W * H, dtype=np.int32), 0, 1)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    finally:
        ctx.close()
        orc.close()
