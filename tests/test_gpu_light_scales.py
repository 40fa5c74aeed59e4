"""Light-tree choices at sizes where the short reciprocal, quotient and root
of the importance do not hold (the descent then takes the general ones), and
at the sizes where they do: the light chosen at every first hit is the
oracle's."""
import math

import numpy as np
import pytest

import oracle_binding as ob
from psycles_amd import abi, scenes
from psycles_amd.render import RendererBackend

pytestmark = pytest.mark.gpu


def lit_floor(scale, flat):
    """A floor under 60 emissive triangles of very different sizes; `flat`
    collapses a third of them to points, whose extent is zero."""
    rng = np.random.RandomState(8)
    p, t = scenes.quad([[-1, 0, -1], [-1, 0, 1], [1, 0, 1], [1, 0, -1]])
    floor = scenes.MeshData((p * scale).astype(np.float32), t, [0])
    centre = rng.uniform((-1, 0.1, -1), (1, 1.5, 1), (60, 1, 3))
    size = 10.0 ** rng.uniform(-3, -0.7, (60, 1, 1))
    corners = centre + size * rng.uniform(-1, 1, (60, 3, 3))
    if flat:
        corners[::3] = centre[::3] + 1e-9 * rng.uniform(-1, 1, (20, 3, 3))
    glow = scenes.MeshData((corners.reshape(-1, 3) * scale).astype(np.float32),
                           np.arange(180, dtype=np.uint32).reshape(-1, 3), [1])
    materials = [scenes.diffuse_material((0.7, 0.7, 0.7)), scenes.emission_material((1, 1, 1), 5.0)]
    camera = scenes.CameraData(scenes.look_at((0.0, 2.0 * scale, 2.5 * scale), (0.0, 0.0, 0.0)), math.radians(50.0),
                               1.0e-3 * scale, 100.0 * scale)
    snap = scenes.SceneSnapshot(materials, [floor, glow],
                                [scenes.InstanceData(0, scenes.identity()), scenes.InstanceData(1, scenes.identity())],
                                camera, name="lit floor")
    snap.lights = [scenes.lamp(abi.LIGHT_POINT, scenes.translation(0.3 * scale, 0.8 * scale, 0.1 * scale), power=3.0,
                               size=0.0),
                   scenes.lamp(abi.LIGHT_DISTANT, scenes.frame_z((0.2, 1.0, 0.4)), power=1.0, angle=0.1)]
    return snap


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("scale", [1.0e-7, 1.0e-3, 1.0, 1.0e4, 2.0e9])
def test_light_choice(scale, flat):
    print(f"case: light choice at scale {scale}, flat {flat}", flush=True)
    snap = lit_floor(scale, flat)
    s = scenes.many_light_settings(72, 48)
    backend = RendererBackend(0)
    scene = backend.compile_scene(snap).scene
    session = backend.create_session(scene, s)
    oracle = ob.OracleScene(snap)
    chosen = set()
    for sample in (0, 5):
        a = session.trace_events(sample, 16)[:, :, 0]
        b = oracle.trace_events(s, sample, 16)[:, :, 0]
        for word in (abi.TRACE_FLAGS, abi.TRACE_OBJECT, abi.TRACE_PRIMITIVE, abi.TRACE_LIGHT):
            assert np.array_equal(a[..., word] & 31 if word == abi.TRACE_FLAGS else a[..., word],
                                  b[..., word] & 31 if word == abi.TRACE_FLAGS else b[..., word]), word
        chosen |= set(np.unique(b[..., abi.TRACE_LIGHT]).tolist())
    assert len(chosen) > 10
    session.close()
    scene.close()
    backend.close()


def lamps_over_floor(scale):
    """A floor under 24 point lamps without extent, the nearest of them at
    half a scale: their square distances span a factor of 64."""
    rng = np.random.RandomState(4)
    p, t = scenes.quad([[-1, 0, -1], [-1, 0, 1], [1, 0, 1], [1, 0, -1]])
    floor = scenes.MeshData((p * scale).astype(np.float32), t, [0])
    camera = scenes.CameraData(scenes.look_at((0.0, 2.0 * scale, 2.5 * scale), (0.0, 0.0, 0.0)), math.radians(50.0),
                               1.0e-3 * scale, 100.0 * scale)
    snap = scenes.SceneSnapshot([scenes.diffuse_material((0.7, 0.7, 0.7))], [floor],
                                [scenes.InstanceData(0, scenes.identity())], camera, name="lamps over a floor")
    snap.lights = [scenes.lamp(abi.LIGHT_POINT, scenes.translation(*(scale * np.array([x, y, z]))), power=3.0, size=0.0)
                   for x, y, z in rng.uniform((-1, 0.5, -1), (1, 3.0, 1), (24, 3))]
    return snap


# square distances of 2^-60 lie within the second to fourth of these
@pytest.mark.parametrize("scale", [2.0e-10, 3.0e-10, 6.0e-10, 1.0e-9, 3.0e-9])
def test_light_choice_at_the_least_distances(scale):
    print(f"case: light choice over lamps at scale {scale}", flush=True)
    snap = lamps_over_floor(scale)
    s = scenes.many_light_settings(72, 48)
    backend = RendererBackend(0)
    scene = backend.compile_scene(snap).scene
    session = backend.create_session(scene, s)
    oracle = ob.OracleScene(snap)
    chosen = set()
    for sample in (0, 5):
        a = session.trace_events(sample, 16)[:, :, 0]
        b = oracle.trace_events(s, sample, 16)[:, :, 0]
        for word in (abi.TRACE_FLAGS, abi.TRACE_OBJECT, abi.TRACE_PRIMITIVE, abi.TRACE_LIGHT):
            assert np.array_equal(a[..., word] & 31 if word == abi.TRACE_FLAGS else a[..., word],
                                  b[..., word] & 31 if word == abi.TRACE_FLAGS else b[..., word]), word
        chosen |= set(np.unique(b[..., abi.TRACE_LIGHT]).tolist())
    assert len(chosen) > 10
    session.close()
    scene.close()
    backend.close()
