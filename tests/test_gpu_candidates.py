"""Light candidates at the edges of the mid-range arithmetic (area_candidate
and phat, csrc/vr_kernels.hip and vr_device.h): emission so small or so large
that targets leave the range where the short square roots and quotients are
exact, emitters up to half the map that shading points lie inside of, beside
and touching, and emitters at the map's corner.  The general path takes over
there, so every output equals the oracle's bit for bit."""
import dataclasses

import numpy as np
import pytest

from _parity import run_config
from smallproject_amd import _lib, configs

pytestmark = pytest.mark.gpu


def _odd_lights(world, renderer):
    L = world.lights()
    rng = np.random.default_rng(3)
    n = len(L)
    L["size"] = rng.choice([1, 1, 2, 8, 63, 512], n)
    x, y, z = (rng.integers(0, 160, n) for _ in range(3))
    x[::5], y[::7], z[::3] = 0, 0, 0
    at = np.arange(n) % 4 == 3  # some stay where the scene put them
    pos = (x + z * 1024 + y * 1024 * 1024).astype(np.uint32)
    L["position"] = np.where(at, L["position"], pos)
    world.setup_light_buffer(L)
    renderer.set_lights(L)


@pytest.mark.parametrize("point", [False, True])
@pytest.mark.parametrize("source", [_lib.SOURCE_UNIFORM, _lib.SOURCE_POWER])
@pytest.mark.parametrize("lut", [(1e-36, 1e-30), (1e-12, 1e12), (1e18, 1e24)])
def test_candidates_at_the_edges(gpu, point, source, lut):
    sc = dataclasses.replace(configs.CONFIGS["c1_point_128"], point=point, lut=lut, emit_range=(1, 255), lights=256)
    for flags in (0, _lib.FLAG_MIS_SPATIAL):
        res = run_config(sc, frames=2, width=150, height=90, source=source, flags=flags, setup=_odd_lights)
        report = "\n".join(c.report() for c in res)
        assert all(c.ok for c in res), f"point {point} source {source} lut {lut} flags {flags}\n{report}"
