"""Scenes whose instance BVH is one leaf start their rays on the mesh's root,
in builds of their own; scenes of several untransformed instances, or of one
with a transform, walk to it.  All give the records and the visit counts of
the one-lane grid kernel, which always walks."""

import numpy as np
import pytest

from psychopath_amd import scenes
from psychopath_amd.tracer import Assembly, DeviceHitRecords, DeviceRays, Mesh, RayBatch, Tracer

pytestmark = pytest.mark.gpu

# (kernel, waves_per_cu, refill_min, stack_lds, simd_waves, leaf_min)
SHAPES = ((0, 24, 16, 16, 4, 32), (0, 16, 16, 8, 8, 16), (0, 8, 8, 24, 4, 0), (0, 16, 16, 24, 8, 32),
          (2, 16, 16, 16, 4, 16), (2, 8, 8, 8, 8, 0))


@pytest.mark.parametrize("instances,samples", [(0, 1), (1, 1), (1, 2), (2, 1), (2, 3), (5, 1), ("moved", 1)])
def test_one_leaf_and_walked_scenes_agree(instances, samples):
    v, f = scenes.displaced_sphere(4)
    asm = Assembly()
    count = 1 if instances == "moved" else instances
    for part in np.array_split(np.arange(len(f)), max(1, count)):
        w = v if samples == 1 else np.stack([v * np.float32(1 + 0.1 * k) for k in range(samples)])
        asm.add_mesh(Mesh(w, f[part]))
    for k in range(count):
        asm.add_instance(k, scenes.translate_xf((0.1, 0.0, 0.2))[None] if instances == "moved" else None)
    tracer = Tracer(asm.build(), max_batch=1 << 14)
    r = scenes.incoherent_rays(v.min(0), v.max(0), 5001, seeds=(41, 42, 43))
    occ = (np.arange(5001) % 4 == 0).astype(np.uint8)
    rays = DeviceRays(RayBatch(*(r[k] for k in ("ox", "oy", "oz", "dx", "dy", "dz", "time", "max_t")), occ))

    def go(shape):
        tracer.set_tuning(*shape)
        hits, counted = DeviceHitRecords(rays.n), DeviceHitRecords(rays.n)
        tracer.trace_device(rays, hits)
        visits = tracer.trace_counted(rays, counted)
        assert hits.records().tobytes() == counted.records().tobytes()
        return hits.records(), visits

    want, visits = go((1, 1, 1, 8, 4, 0))
    assert (want["kind"] == 2).sum() > 1000 or not count
    for shape in SHAPES:
        got, counts = go(shape)
        assert got.tobytes() == want.tobytes() and counts == visits, shape
