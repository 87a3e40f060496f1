"""The persistent kernels' two box tests: rays and scenes that the reduced
test of finite rays does not serve (zero direction components, origins in a
box's planes, infinities, NaN) and, in the same waves, rays that it does,
must give the records of the one-lane grid kernel, which has the reference's
box test only; on the static scene without NaN also the oracle's.  Scenes
whose boxes the reduced test does not serve (NaN, empty, or infinite where
they are lerped) must take the full one."""

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


def odd_scene(kind):
    """A plain instance beside one whose box in the instance BVH, or in a
    time-sampled node, is empty ([+inf, -inf]) or infinite."""
    v, f = steps_mesh()
    place = np.array([[1, 0, 0, -3, 0, 1, 0, 0, 0, 0, 1, -6]], np.float32)
    flat = np.array([[1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 0, 0]], np.float32)
    meshes, instances = [(v, f)], [(0, None)]
    if kind == "flattened":
        instances.append((0, flat))
    elif kind == "flattened, moving":
        instances.append((0, np.concatenate([flat, flat + np.eye(1, 12, 3, dtype=np.float32)])))
    elif kind == "scaled to nothing":
        instances.append((0, np.zeros((1, 12), np.float32)))
    elif kind == "one leaf with a NaN vertex":
        w = np.array([(2, 2, 6), (9, 2, 6), (2, 9, 6), (3, 3, 7), (8, 3, 7), (np.nan,) * 3], np.float32)
        meshes.append((w, np.array([(0, 1, 2), (3, 4, 5)], np.uint32)))
        instances.append((1, place))
    elif kind == "all NaN":
        meshes.append((np.full((3, 3), np.nan, np.float32), np.array([(0, 1, 2)], np.uint32)))
        instances.append((1, place))
    elif kind == "both infinities":
        w = v.copy()
        w[5], w[90] = np.inf, -np.inf
        meshes.append((w, f))
        instances.append((1, place))
    else:  # infinite planes in time samples
        w = np.stack([v, v + 1])
        w[0, 5], w[1, 90], w[:, 200] = np.inf, -np.inf, np.inf
        meshes.append((w, f))
        instances.append((1, None))
    return meshes, instances


@pytest.mark.parametrize("kind", ["flattened", "flattened, moving", "scaled to nothing", "one leaf with a NaN vertex",
                                  "all NaN", "both infinities", "infinite, moving"])
def test_odd_boxes_take_the_full_test(kind):
    from oracle.psyref import OracleScene
    meshes, instances = odd_scene(kind)
    a, o = Assembly(), OracleScene()
    for m in meshes:
        a.add_mesh(Mesh(*m))
        o.add_mesh(*m)
    for mesh, xf in instances:
        a.add_instance(mesh, xf)
        o.add_instance(mesh, xf)
    o.build()
    tracer = Tracer(a.build(), max_batch=1 << 14)
    # All kinds of rays, then finite ones only, in whole waves of their own:
    # no lane of these forces the full test on the others.
    batch = rays()
    rng = np.random.default_rng(6)
    n = 4096
    p, q = (rng.uniform(-1, 13, (n, 3)).astype(np.float32) for _ in range(2))
    t = (np.arange(n) % 3 / 2).astype(np.float32)
    fields = [np.concatenate(x) for x in zip((getattr(batch, k) for k in ("ox", "oy", "oz", "dx", "dy", "dz", "time",
                                                                           "max_t")),
                                             (*p.T, *(q - p).T, t, np.full(n, np.inf, np.float32)))]
    batch = RayBatch(*fields, np.concatenate([batch.flags, np.zeros(n, np.uint8)]))
    dr = DeviceRays(batch)
    want = records(tracer, (1, 1, 1, 8, 4, 0), dr)
    w = o.trace({k: getattr(batch, k) for k in ("ox", "oy", "oz", "dx", "dy", "dz", "time", "max_t")}
                | {"occlusion": batch.flags})
    finite = slice(len(batch) - n, None)
    assert np.array_equal(want["kind"][finite], w["kind"][finite])
    # (which hit a ray ends on that met a NaN one is not defined)
    s = (w["kind"] == 2) & np.isfinite(w["t"]) & np.isfinite(want["t"])
    s[:finite.start] = False
    for k in ("t", "prim_id", "inst_id"):
        assert np.array_equal(want[k][s], w[k][s]), k
    alone = DeviceRays(batch.slice(finite.start, len(batch)))
    tracer.set_tuning(1, 1, 1, 8, 4, 0)
    visits = tracer.trace_counted(alone, DeviceHitRecords(n))
    assert visits["instance_visits"] > n
    for shape in SHAPES:
        assert records(tracer, shape, dr).tobytes() == want.tobytes(), (kind, shape)
        assert records(tracer, shape, alone).tobytes() == want[finite].tobytes(), (kind, shape)
        assert tracer.trace_counted(alone, DeviceHitRecords(n)) == visits, (kind, shape)
