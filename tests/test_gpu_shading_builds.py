"""The shading kernels' builds by register budget, in the wavefront and the
one-launch form, sorted and not, give the same image bit for bit on scenes
that between them have every closure, light kind and time-sampled input."""

import numpy as np
import pytest

from psychopath_amd import render, scenes

pytestmark = pytest.mark.gpu


def every_closure():
    sc = scenes.cornell_box(64, 64, 4, 4, 5)
    sc.shaders.append((scenes.SHADER_DIELECTRIC, scenes.rec709(0.95, 0.95, 0.95), 0.1, 1.5))
    sc.shaders.append((scenes.SHADER_GGX, scenes.rec709(0.9, 0.8, 0.4), 0.3, 0.8))
    sc.shaders.append((scenes.SHADER_EMIT, scenes.rec709(0.5, 0.5, 0.5), 0.0, 0.0))
    sc.instances[5]["shader"] = 3
    sc.instances[6]["shader"] = 4
    sc.instances[2]["shader"] = 5
    sc.instances[3]["shader"] = None  # emits the colour of surfaces without a shader
    sc.sphere_lights.append((0.3, [scenes.rec709(20, 10, 5), scenes.rec709(5, 10, 20)]))
    sc.instances.append(dict(kind="sphere", index=0, shader=None, xforms=scenes.translate_xf((-2.0, 2.0, 2.0))[None]))
    return sc


SCENES = {
    "every closure": every_closure,
    "cornell": lambda: scenes.cornell_box(64, 64, 4, 4, 5),
    "smooth sphere": lambda: scenes.sphere_scene(5, smooth=True),
    "moving instances": lambda: scenes.motion_instances(grid=4, levels=4),
    "nested lights": scenes.nested_lights_scene,
    "metal, glass and emitters": lambda: scenes.large_scene(grid=8, lights=32),
    "distant light": lambda: scenes.terrain_scene(64, 40),
}


@pytest.mark.parametrize("name", sorted(SCENES))
def test_all_builds_agree(name):
    sc = SCENES[name]()
    r = render.build(sc)
    st = dict(width=64, height=64, spp=4, max_bounces=4, seed=3)
    want, stats = r.render(sc.camera, st)
    assert want.max() > 0
    for waves in (1, 2, 3, 4):
        for opt in (dict(sort=True), dict(sort=False), dict(plain=True)):
            r.set_options(shade_waves=waves, **opt)
            img, s = r.render(sc.camera, st)
            assert s["rays"] == stats["rays"], (waves, opt)
            assert np.array_equal(img, want), (waves, opt)
