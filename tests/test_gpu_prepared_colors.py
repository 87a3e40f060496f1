"""Colours a renderer lays out once (shaders, background, lights without time
samples) and those it evaluates from the shared tables (lights with colour
samples, lights and shaders beyond the first 4,096): renders match the oracle's
for colours in inner and border cells of the upsampling grid, outside it, and
black, and what a renderer lays out stays bounded."""

import ctypes as C

import numpy as np
import pytest

from psychopath_amd import _lib, render, scenes
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


@pytest.mark.parametrize("kind", ["xyz", "blackbody"])
def test_unused_shaders_take_no_memory(kind):
    """A shader record is 32 bytes; 200,000 colours laid out would be 300 MB."""
    def free():
        f, total = C.c_size_t(), C.c_size_t()
        assert _lib.lib().hipMemGetInfo(C.byref(f), C.byref(total)) == 0  # (of the runtime the library runs on)
        return f.value

    sc = scenes.cornell_box(16, 16, 1, 1, 0)
    sc.shaders += [(scenes.SHADER_LAMBERT, (XYZ, 0.2, 0.3, 0.4) if kind == "xyz" else (BLACKBODY, 4000.0, 1e-9, 0.0),
                    0.0, 0.0)] * 200_000
    render.build(sc, 4096)  # what a first renderer loads stays
    before = free()
    r = render.build(sc, 4096)
    used = before - free()
    r.render(sc.camera, sc.settings)
    # the scene, 4,096 paths, 200,000 records and 2 * 4,096 colours are some
    # 25 MB, in allocations of 2 MB
    assert used < 80 << 20, used


def test_shaders_beyond_the_prepared_ones_match_oracle():
    sc = scenes.cornell_box(24, 24, 4, 3, 0)
    first = [(scenes.SHADER_LAMBERT, (XYZ, 0.01 * (k % 50), 0.3, 0.2), 0.0, 0.0) for k in range(4095)]
    for inst in sc.instances:
        if inst.get("shader"):
            inst["shader"] += len(first)
    sc.shaders = sc.shaders[:1] + first + sc.shaders[1:]
    check_parity(sc, "4,098 shaders")
