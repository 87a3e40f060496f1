"""The persistent kernels' two box tests: rays and scenes that the reduced
test of finite rays does not serve (zero direction components, origins in a
box's planes, infinities, NaN) and, in the same waves, rays that it does,
must give the records of the one-lane grid kernel, which has the reference's
box test only; on the static scene without NaN also the oracle's."""

import numpy as np
import pytest

from psychopath_amd.tracer import Assembly, DeviceHitRecords, DeviceRays, Mesh, RayBatch, Tracer

pytestmark = pytest.mark.gpu

# (kernel, waves_per_cu, refill_min, stack_lds, simd_waves, leaf_min)
SHAPES = ((0, 16, 16, 16, 4, 0), (0, 4, 1, 8, 8, 8), (0, 24, 16, 24, 4, 32), (2, 8, 16, 8, 4, 16))


def steps_mesh(nan=False):
    """A staircase of axis-aligned quads on integer coordinates: flat boxes
    whose planes rays and origins lie in."""
    verts, tris = [], []
    for x in range(12):
        for y in range(12):
            z = (x * y) % 5
            b = len(verts)
            verts += [(x, y, z), (x + 1, y, z), (x + 1, y + 1, z), (x, y + 1, z)]
            tris += [(b, b + 1, b + 2), (b, b + 2, b + 3)]
    v = np.array(verts, np.float32)
    if nan:
        v[77] = np.nan
    return v, np.array(tris, np.uint32)


def rays():
    rng = np.random.default_rng(5)
    n = 3000
    o = rng.integers(-1, 13, (n, 3)).astype(np.float32)
    o[::3] += rng.random((len(o[::3]), 3), dtype=np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    axis = np.eye(3, dtype=np.float32)[rng.integers(0, 3, n)] * rng.choice([-1.0, 1.0], n).astype(np.float32)[:, None]
    d[::2] = axis[::2]
    d[1::8, 0] = -0.0
    max_t = np.full(n, np.inf, np.float32)
    max_t[::7] = 4.0
    max_t[5::97] = np.nan
    o[11::101, 1] = np.inf
    o[13::103, 2] = np.nan
    d[17::107, 0] = np.inf
    d[19::109] = 0.0
    occ = (np.arange(n) % 5 == 0).astype(np.uint8)
    t = rng.random(n, dtype=np.float32)
    return RayBatch(*o.T, *d.T, t, max_t, occ)


def build(kind):
    v, f = steps_mesh(nan=kind == "nan")
    if kind == "motion":
        v = np.stack([v, v + np.float32(0.5) * (np.arange(len(v)) % 3 == 0)[:, None].astype(np.float32)])
    a = Assembly()
    a.add_mesh(Mesh(v, f))
    quarter = np.array([[0, 1, 0, 0, -1, 0, 0, 12, 0, 0, 1, -2]], np.float32)
    moved = np.array([[1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 3], [1, 0, 0, 1, 0, 1, 0, 0, 0, 0, 1, 4]], np.float32)
    a.add_instance(0)
    if kind == "xform":
        a.add_instance(0, quarter)
    if kind == "motion":
        a.add_instance(0, moved)
    return a.build(), v, f


def records(tracer, shape, dr):
    tracer.set_tuning(*shape)
    hits = DeviceHitRecords(dr.n)
    hits.buf.upload(np.full(dr.n * 32, 0xFF, np.uint8))
    tracer.trace_device(dr, hits)
    return hits.records()


@pytest.mark.parametrize("kind", ["static", "xform", "motion", "nan"])
def test_box_tests_agree(kind):
    scene, v, f = build(kind)
    tracer = Tracer(scene, max_batch=1 << 14)
    batch = rays()
    dr = DeviceRays(batch)
    want = records(tracer, (1, 1, 1, 8, 4, 0), dr)
    assert 200 < (want["kind"] == 2).sum() and (want["kind"] == 1).sum() > 20
    for shape in SHAPES:
        got = records(tracer, shape, dr)
        assert got.tobytes() == want.tobytes(), (kind, shape)
    if kind == "static":
        from oracle.psyref import OracleScene
        o = OracleScene()
        o.add_mesh(v, f)
        o.add_instance(0)
        o.build()
        w = o.trace({k: getattr(batch, k) for k in ("ox", "oy", "oz", "dx", "dy", "dz", "time", "max_t")}
                    | {"occlusion": batch.flags})
        assert np.array_equal(want["kind"], w["kind"])
        s = (w["kind"] == 2) & np.isfinite(w["t"])  # (a NaN hit of a NaN ray: which of many is not defined)
        for k in ("t", "b0", "b1", "b2", "prim_id"):
            assert np.array_equal(want[k][s], w[k][s]), k
