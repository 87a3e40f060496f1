"""How the persistent kernels deal the rays of a launch to their waves: below
one ray per lane every wave starts on an even share and no counter is read,
above it the rest comes from eight counters.  Around the sizes where that
changes, and where a range's last block is cut, every record is written once
and equals the one-lane grid kernel's."""

import numpy as np
import pytest

from psychopath_amd import scenes
from psychopath_amd.tracer import Assembly, DeviceHitRecords, DeviceRays, Mesh, RayBatch, Tracer

pytestmark = pytest.mark.gpu

LANES = 256 * 64  # of one wave on each of the 256 compute units
SIZES = (1, 7, 8, 9, 511, 512, 513, 2048, LANES - 1, LANES, LANES + 1, LANES + 512, LANES + 513, 2 * LANES + 63,
         3 * LANES - 65)


@pytest.fixture(scope="module")
def traced():
    v, f = scenes.displaced_sphere(4)
    a = Assembly()
    a.add_mesh(Mesh(v, f))
    a.add_instance(0)
    tracer = Tracer(a.build(), max_batch=1 << 16)
    r = scenes.incoherent_rays(v.min(0), v.max(0), max(SIZES), seeds=(171, 172, 173))
    tracer.set_tuning(1, 1, 1, 8, 4, 0)
    return tracer, r, records(tracer, batch(r, max(SIZES)))


def batch(r, n):
    return DeviceRays(RayBatch(*(r[k][:n] for k in ("ox", "oy", "oz", "dx", "dy", "dz", "time", "max_t"))))


def records(tracer, rays):
    hits = DeviceHitRecords(rays.n)
    hits.buf.upload(np.full(rays.n * 32, 0xFF, np.uint8))
    tracer.trace_device(rays, hits)
    return hits.records()


@pytest.mark.parametrize("n", SIZES)
def test_every_ray_is_dealt_once(traced, n):
    tracer, r, want = traced
    rays = batch(r, n)
    for shape in ((0, 1, 1, 16, 4, 0), (0, 1, 64, 8, 8, 32), (0, 2, 16, 16, 4, 16), (2, 1, 16, 16, 4, 16)):
        tracer.set_tuning(*shape)
        assert records(tracer, rays).tobytes() == want[:n].tobytes(), (n, shape)
