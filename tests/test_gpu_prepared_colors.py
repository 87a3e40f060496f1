"""Colours a renderer lays out once (shaders, background, lights without time
samples) and those it evaluates from the shared tables (lights with colour
samples or beyond the first 4,096): renders match the oracle's for colours in
inner and border cells of the upsampling grid, outside it, and black."""

import numpy as np
import pytest

from psychopath_amd import scenes
from tests.test_gpu_render import check_parity

pytestmark = pytest.mark.gpu

XYZ, BLACKBODY = scenes.COLOR_XYZ, scenes.COLOR_BLACKBODY
COLOURS = {
    "inner": (XYZ, 0.5, 0.45, 0.4, ),
    "red edge": scenes.rec709(0.9, 0.0, 0.0),
    "blue edge": scenes.rec709(0.0, 0.0, 0.9),
    "near the locus": (XYZ, 0.72, 0.27, 0.0),
    "outside": (XYZ, 1.0, 0.0, 0.0),
    "black": (XYZ, 0.0, 0.0, 0.0),
    "no sum": (XYZ, 0.5, -0.5, 0.0),
}


@pytest.mark.parametrize("name", sorted(COLOURS))
def test_shader_and_light_colours_match_oracle(name):
    sc = scenes.cornell_box(24, 24, 4, 3, 0)
    sc.shaders[1] = (scenes.SHADER_LAMBERT, COLOURS[name], 0.0, 0.0)
    sc.shaders[2] = (scenes.SHADER_GGX, COLOURS[name], 0.3, 0.5)
    sc.background = COLOURS[name]
    kind, x, y, z = COLOURS[name]
    sc.rect_lights[0] = (0.25, 0.25, (kind, 80 * x, 80 * y, 80 * z))
    check_parity(sc, name)


@pytest.mark.parametrize("lights", [3, 4200])
def test_sphere_light_colours_match_oracle(lights):
    sc = scenes.cornell_box(24, 24, 2, 2, 0)
    rng = np.random.default_rng(11)
    for k in range(lights):
        c = scenes.rec709(*(rng.random(3) * 40))
        if k % 3 == 1:
            c = [c, scenes.rec709(*(rng.random(3) * 40))]  # two time samples
        if k % 3 == 2:
            c = (BLACKBODY, float(rng.uniform(2500, 9000)), 1e-9, 0.0)
        sc.sphere_lights.append((0.03, c))
        pos = rng.uniform((-5.0, 0.5, 0.5), (-0.5, 5.0, 5.0))
        sc.instances.append(dict(kind="sphere", index=k, shader=None, xforms=scenes.translate_xf(pos)[None]))
    check_parity(sc, f"{lights} sphere lights")
