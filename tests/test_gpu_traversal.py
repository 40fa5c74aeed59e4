"""The phased traversal against the oracle where its bookkeeping can go wrong.

Waves that are partly filled, stacks deeper than the LDS ring (entries spill
to HBM and come back), lanes that enter, leave and skip instances while
others are inside one, single-user meshes in and outside the world tree,
rays with NaN.  Closest hits identical, shadow
transmittance bit-identical.
"""
import ctypes as C
import sys

import numpy as np
import pytest

import oracle_binding as ob
from psycles_amd import abi, scenes
from psycles_amd.render import RendererBackend

pytestmark = pytest.mark.gpu


def heap_of_triangles(count=3000, seed=11):
    """Large triangles through one ball: no split separates them, so a ray
    visits most of the tree and its stack grows past the LDS ring."""
    rng = np.random.RandomState(seed)
    p = rng.uniform(-1.0, 1.0, (3 * count, 3)).astype(np.float32)
    t = np.arange(3 * count, dtype=np.uint32).reshape(-1, 3)
    return scenes.MeshData(p, t, [0])


def mixed_scene():
    """Triangle heaps shared by overlapping instances of different
    visibility, one single-user mesh and a floor; opaque and part
    transparent materials."""
    rng = np.random.RandomState(5)
    small = heap_of_triangles(40, 3)
    ball_p, ball_t = scenes.geodesic_icosphere(4)
    fp, ft = scenes.quad([[-6, -2, -6], [-6, -2, 6], [6, -2, 6], [6, -2, -6]])
    meshes = [small, scenes.MeshData(ball_p, ball_t, [0]), scenes.MeshData(fp, ft, [1]), heap_of_triangles(60, 4),
              heap_of_triangles(50, 6)]
    materials = [scenes.mix_diffuse_transparent((0.5, 0.6, 0.7), 0.7), scenes.diffuse_material((0.5, 0.5, 0.5))]
    instances = []
    for k in range(24):
        m = scenes.translation(*rng.uniform(-2.5, 2.5, 3)) @ scenes.rotation_y(float(rng.uniform(0, 360)))
        instances.append(scenes.InstanceData(k % 2, m, material_overrides=[k % 3 == 0],
                                             visibility=[abi.VIS_ALL, abi.VIS_SHADOW, abi.VIS_ALL & ~abi.VIS_SHADOW][k % 3]))
    # single-user meshes: with a plain mask and with all bits set they join
    # the world tree, with other bits they keep a tree of their own
    instances += [scenes.InstanceData(2, scenes.identity()),
                  scenes.InstanceData(3, scenes.translation(0.5, 0.0, 0.5), visibility=0xffffffff),
                  scenes.InstanceData(4, scenes.translation(-0.5, 0.3, 0.0), visibility=0x50)]
    camera = scenes.CameraData(scenes.translation(0, 0, 6))
    return scenes.SceneSnapshot(materials, meshes, instances, camera, name="mixed")


def heap_scene():
    camera = scenes.CameraData(scenes.translation(0, 0, 4))
    return scenes.SceneSnapshot([scenes.mix_diffuse_transparent((0.5, 0.5, 0.5), 0.9)], [heap_of_triangles()],
                                [scenes.InstanceData(0, scenes.identity())], camera, name="heap")


def nested_scales():
    """Three meshes of triangles whose sizes fall by powers of two, each mesh
    every third power.  One tree over all of them has about 22 levels of four,
    too many for the traversal stack, so each mesh keeps its own (about 12)."""
    meshes = []
    for m in range(3):
        sizes = 2.0 ** (60.0 - np.arange(m, 131, 3))
        corners = np.array([[1.0, 1.0, 1.0], [1.3, 1.0, 1.15], [1.1, 1.3, 1.3]])
        p = (sizes[:, None, None] * corners[None]).reshape(-1, 3).astype(np.float32)
        meshes.append(scenes.MeshData(p, np.arange(len(p), dtype=np.uint32).reshape(-1, 3), [0]))
    return scenes.SceneSnapshot([scenes.diffuse_material((0.5, 0.5, 0.5))], meshes,
                                [scenes.InstanceData(m, scenes.identity()) for m in range(3)],
                                scenes.CameraData(scenes.translation(0, 0, 4)), name="scales")


SCENES = {"heap": (heap_scene, 1.5), "mixed": (mixed_scene, 4.0), "scales": (nested_scales, 2.0)}


def queries(n, reach, seed, kind):
    rng = np.random.RandomState(seed)
    out = []
    for i in range(n):
        a, b = rng.uniform(-reach, reach, 3), rng.uniform(-reach, reach, 3)
        d = (b - a) / np.linalg.norm(b - a)
        q = {"origin": a, "direction": d, "kind": kind, "tmin": float(rng.choice([0.0, 0.1])),
             "tmax": float(rng.choice([0.5, 100.0])), "transparent_max": 40}
        q["visibility"] = (abi.VIS_SHADOW if kind == abi.QUERY_SHADOW
                           else int(rng.choice([abi.VIS_ALL, abi.VIS_CAMERA, 0x40])))
        if i % 13 == 5:
            q["direction"] = [0.0, 1.0, 0.0]
        if i % 3 == 1:  # a ray near the diagonal, where the scales are nested
            b = np.ones(3) * rng.uniform(0.9, 1.5) + rng.uniform(0.0, 0.3, 3)
            q["origin"], q["direction"] = b * 2.0 ** rng.randint(-8, 8), -b / np.linalg.norm(b) + rng.uniform(-0.1, 0.1, 3)
        if i % 17 == 3:
            q["origin"] = [a[0], float("nan"), a[2]]
        out.append(q)
    return out


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1500])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_queries_match_oracle(name, n):
    print(f"case: traversal of {name}, {n} queries", flush=True)
    sys.stdout.flush()
    make, reach = SCENES[name]
    snap = make()
    backend = RendererBackend(0)
    dev = backend.compile_scene(snap).scene
    ora = ob.OracleScene(snap)
    closest = queries(n, reach, 100 + n, abi.QUERY_CLOSEST)
    for x, y in zip(dev.intersect(closest), ora.intersect(closest)):
        assert (x.hit, x.object, x.primitive) == (y.hit, y.object, y.primitive)
        if x.hit:
            assert np.float32([x.t, x.u, x.v]).tobytes() == np.float32([y.t, y.u, y.v]).tobytes()
    shadow = queries(n, reach, 200 + n, abi.QUERY_SHADOW)
    for x, y in zip(dev.intersect(shadow), ora.intersect(shadow)):
        assert np.float32(x.transmittance).tobytes() == np.float32(y.transmittance).tobytes()
        assert x.hit == y.hit
    dev.close()
    backend.close()


@pytest.mark.parametrize("width,height,spp", [(1, 1, 1), (8, 8, 1), (17, 3, 2), (64, 64, 1), (257, 129, 3), (640, 400, 9)])
def test_short_queues(width, height, spp):
    """Queues from one entry to several reservations a wave (4096 waves, 64 to
    256 entries each): the trace kernel deals them out; film and ray count are
    those of the one-lane-per-path kernel."""
    print(f"case: short queues {width}x{height}x{spp}", flush=True)
    snap = scenes.cornell_lamps()
    films = []
    for integrator in (abi.INTEGRATOR_MEGAKERNEL, abi.INTEGRATOR_WAVEFRONT):
        backend = RendererBackend(0, integrator=integrator, max_samples_per_dispatch=spp)
        scene = backend.compile_scene(snap).scene
        session = backend.create_session(scene, scenes.cornell_settings(width, height))
        session.render_device(0, spp, spp)
        films.append([a.tobytes() for a in session.read_film()] + [session.stats().rays])
        session.close()
        scene.close()
        backend.close()
    assert films[0] == films[1]


@pytest.mark.parametrize("shape", [
    {"trace_chunk": 16, "refill_lanes": 1}, {"trace_chunk": 16, "refill_lanes": 64, "list_chunk": 64},
    {"trace_chunk": 4096, "list_chunk": 256}, {"queue_chunk": 128, "list_chunk": 256}])
def test_long_queues_of_other_shapes(shape):
    """Reservations of 32 to 8192 queue entries and 128 to 512 list entries,
    on queues that hold many of the small ones and fewer than one of the large
    ones a wave: film and ray count are those of the default shape."""
    print(f"case: long queues, {shape}", flush=True)
    backend = RendererBackend(0, integrator=abi.INTEGRATOR_WAVEFRONT, max_samples_per_dispatch=3)
    scene = backend.compile_scene(scenes.cornell_lamps()).scene
    films = []
    for tuning in ({}, shape):
        session = backend.create_session(scene, scenes.cornell_settings(643, 401))
        if tuning:
            session.set_tuning(tuning)
        session.render_device(0, 3, 3)
        films.append([a.tobytes() for a in session.read_film()] + [session.stats().rays])
        session.close()
    assert films[0] == films[1]
    scene.close()
    backend.close()


@pytest.mark.parametrize("n", [1, 65, 4099, 300001])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_mixed_queries(name, n):
    """Closest hits and shadows in one call, from one query to more than the
    waves of a full launch reserve at first (262144): every word of every hit
    is the oracle's, also where a lane answers several queries in turn."""
    print(f"case: mixed queries of {name}, {n} queries", flush=True)
    make, reach = SCENES[name]
    snap = make()
    backend = RendererBackend(0)
    dev = backend.compile_scene(snap).scene
    ora = ob.OracleScene(snap)
    some = [q for pair in zip(queries(300, reach, 5, abi.QUERY_CLOSEST), queries(300, reach, 6, abi.QUERY_SHADOW))
            for q in pair]
    rng = np.random.RandomState(n)
    for q in some:
        q["transparent_max"] = int(rng.choice([0, 1, 2, 40]))
        q["transparent_depth"] = int(rng.choice([0, 1]))
    want = np.frombuffer((abi.RayHit * len(some))(*ora.intersect(some)), np.uint32).reshape(-1, 12)
    records = np.frombuffer(abi.make_queries(some), np.uint32).reshape(-1, 16)
    pick = rng.randint(0, len(some), n)
    sent = np.ascontiguousarray(records[pick])
    got = np.full((n, 12), 0xABABABAB, np.uint32)
    lib = backend.lib
    assert lib.psx_scene_intersect(dev.handle, sent.ctypes.data_as(C.POINTER(abi.RayQuery)), n,
                                   got.ctypes.data_as(C.POINTER(abi.RayHit))) == 0
    shadows = records[pick, 13] == abi.QUERY_SHADOW
    words = [w for w in range(12) if w != 6]  # an early end of a shadow query saves traversals
    assert np.array_equal(got[:, words], want[pick][:, words])
    assert np.array_equal(got[~shadows, 6], want[pick][~shadows, 6])
    assert (got[shadows, 6] >= 1).all() and (got[shadows, 6] <= want[pick][shadows, 6]).all()
    dev.close()
    backend.close()


@pytest.mark.parametrize("kind", [abi.QUERY_CLOSEST, abi.QUERY_SHADOW])
def test_directions_with_nan(kind):
    """A NaN in a direction is the smallest direction of its sign in that
    component, as the clamp of the reference leaves it: the ray is searched."""
    print(f"case: NaN directions, kind {kind}", flush=True)
    snap = heap_scene()
    rays = queries(600, 1.5, 31, kind)
    nan = float("nan")
    for i, q in enumerate(rays):
        d = [float(c) for c in q["direction"]]
        for axis in ((0,), (1,), (2,), (0, 2), (0, 1, 2))[i % 5]:
            d[axis] = nan
        q["direction"] = d
        q["tmax"] = 1.0e30 if i % 5 == 4 else 100.0
        q["tmin"] = 0.0
        if kind == abi.QUERY_CLOSEST:
            q["visibility"] = abi.VIS_ALL
    backend = RendererBackend(0)
    dev = backend.compile_scene(snap).scene
    want = ob.OracleScene(snap).intersect(rays)
    assert 0 < sum(h.hit for h in want)
    for x, y in zip(dev.intersect(rays), want):
        assert (x.hit, x.object, x.primitive) == (y.hit, y.object, y.primitive)
        assert np.float32([x.t, x.u, x.v, *x.transmittance]).tobytes() == \
            np.float32([y.t, y.u, y.v, *y.transmittance]).tobytes()
    dev.close()
    backend.close()
