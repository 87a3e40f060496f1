"""Closest hits sorted by closure kind: around the sizes of a block's tile (4
entries a lane, 16 from 2^20 entries on) the sorted render equals the
unsorted one bit for bit, on a box with every kind of closure."""

import numpy as np
import pytest

from psychopath_amd import render, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(1, 1), (31, 33), (32, 32), (25, 41), (1024, 1023), (1024, 1024), (1111, 1024)])
def test_sorted_render_equals_unsorted(width, height):
    sc = scenes.cornell_box(width, height, 1, 2, 5)
    sc.shaders.append((scenes.SHADER_DIELECTRIC, scenes.rec709(0.95, 0.95, 0.95), 0.1, 1.5))
    sc.shaders.append((scenes.SHADER_GGX, scenes.rec709(0.9, 0.8, 0.4), 0.3, 0.8))
    sc.shaders.append((scenes.SHADER_EMIT, scenes.rec709(0.5, 0.5, 0.5), 0.0, 0.0))
    sc.instances[5]["shader"] = 3
    sc.instances[6]["shader"] = 4
    sc.instances[2]["shader"] = 5
    sc.instances[3]["shader"] = None  # emits the colour of surfaces without a shader
    r = render.build(sc)
    a, sa = r.render(sc.camera, sc.settings)
    r.set_options(sort=False)
    b, sb = r.render(sc.camera, sc.settings)
    assert sa["rays"] == sb["rays"] and (a.max() > 0 or width == 1)
    assert np.array_equal(a, b)
