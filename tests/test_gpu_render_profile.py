"""Profiled and counted renders trace a step's closest-hit and shadow rays in
two launches, ordinary ones in one: the image and the rays are the same, the
profile's rays are the render's, and its visits those of the same rays."""

import numpy as np
import pytest

from psychopath_amd import render, scenes

pytestmark = pytest.mark.gpu

SCENES = {
    "cornell": scenes.cornell_box,
    "moving instances": lambda: scenes.motion_instances(grid=4, levels=4),
    "distant light": lambda: scenes.terrain_scene(64, 40),
}


@pytest.mark.parametrize("bounces", [0, 1, 4])
@pytest.mark.parametrize("max_paths", [0, 3000])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_profiled_and_counted_renders_match(name, max_paths, bounces):
    sc = SCENES[name]()
    r = render.build(sc, max_paths)
    st = dict(width=61, height=47, spp=4, max_bounces=bounces, seed=9)
    want, stats = r.render(sc.camera, st)
    assert want.max() > 0 and (stats["waves"] > 1) == (max_paths != 0)
    visits = []
    for opt in (dict(profile=True), dict(count=True), dict(profile=True, count=True, graphs=False, sort=False)):
        r.set_options(**opt)
        r.profile()
        for _ in range(2):  # (the second sees the counters that the first left)
            img, s = r.render(sc.camera, st)
            p = r.profile()
            assert np.array_equal(img, want), opt
            assert s["rays"] == stats["rays"] and s["paths"] == stats["paths"] == p["paths"], opt
            assert p["closest_rays"] + p["shadow_rays"] == s["rays"] and p["closest_rays"] >= s["paths"], opt
            if "count" in opt:
                visits.append({k: v for k, v in p.items() if k.endswith("visits") or k.endswith("tests")})
            if "profile" in opt:
                assert all(p[k] > 0 for k in ("camera_ms", "trace_ms", "shadow_trace_ms", "shade_ms", "film_ms"))
                assert p["shadow_ms"] == 0
    assert visits[0]["closest_node_visits"] > 0 and all(v == visits[0] for v in visits)
    r.set_options()
    again, s = r.render(sc.camera, st)
    assert np.array_equal(again, want) and s["rays"] == stats["rays"]
