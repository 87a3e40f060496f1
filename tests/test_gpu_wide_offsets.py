"""The traversal builds of scenes above 2^25 nodes (64-bit node offsets),
switched on for small ones: the records and visit counts of the ordinary
builds, and the same renders."""

import numpy as np
import pytest

from psychopath_amd import render, scenes
from psychopath_amd.tracer import Assembly, DeviceHitRecords, DeviceRays, Mesh, RayBatch, Tracer

pytestmark = pytest.mark.gpu


def static(meshes):
    v, f = scenes.displaced_sphere(4)
    asm = Assembly()
    for k, part in enumerate(np.array_split(np.arange(len(f)), meshes)):
        asm.add_mesh(Mesh(v, f[part]))
        asm.add_instance(k)
    return asm


SCENES = {
    "one mesh": lambda: static(1),
    "meshes": lambda: static(3),
    "transforms": lambda: render.assembly_of(scenes.large_scene(grid=4, lights=8)),
    "motion": lambda: render.assembly_of(scenes.motion_instances(grid=4, levels=4)),
    "nested": lambda: render.assembly_of(scenes.nested_lights_scene()),
}


@pytest.mark.parametrize("name", sorted(SCENES))
def test_wide_offsets_give_the_same_records(name):
    scene = SCENES[name]().build()
    tracer = Tracer(scene, max_batch=1 << 14)
    n = 6007
    r = scenes.incoherent_rays((-6, -6, -3), (6, 6, 3), n, seeds=(61, 62, 63))
    occ = (np.arange(n) % 3 == 0).astype(np.uint8)
    fields = [r[k] for k in ("ox", "oy", "oz", "dx", "dy", "dz", "time", "max_t")]
    fields[6] = (np.arange(n) % 11 / 10).astype(np.float32)
    rays = DeviceRays(RayBatch(*fields, occ))

    def go():
        hits, counted = DeviceHitRecords(n), DeviceHitRecords(n)
        tracer.trace_device(rays, hits)
        visits = tracer.trace_counted(rays, counted)
        return hits.records().tobytes(), counted.records().tobytes(), visits

    for shape in ((0, 24, 16, 16, 4, 32), (0, 8, 8, 8, 8, 0), (2, 16, 16, 24, 4, 16)):
        tracer.set_tuning(*shape)
        scene.wide_offsets(False)
        want = go()
        scene.wide_offsets()
        assert go() == want, shape
        assert want[2]["node_visits"] > n or name == "nested"


@pytest.mark.parametrize("make", [scenes.cornell_box, scenes.nested_lights_scene,
                                  lambda: scenes.motion_instances(grid=4, levels=4)])
def test_wide_offsets_give_the_same_image(make):
    sc = make()
    st = dict(width=40, height=33, spp=2, max_bounces=3, seed=2)
    want, _ = render.build(sc).render(sc.camera, st)
    scene = render.assembly_of(sc).build()
    scene.wide_offsets()
    r = render.Renderer(scene, sc.shaders, sc.background, sc.distant_lights)
    got, _ = r.render(sc.camera, st)
    assert want.max() > 0 and np.array_equal(got, want)
