"""Pass pixels and the sampler's table as the device makes them.

The pass kernels' pixels against the same float32 operations on the film's
sums (bit for bit), for every rule and channel count, at pixel counts around
a block's edge; a session that is reset keeps its table only while the sample
total needs the same size; tables of every size against the oracle's sampler.
"""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import oracle_binding as ob
from psycles_amd import abi, scenes
from psycles_amd.render import MemoryOutputSink, RendererBackend, SampleRange, with_passes

pytestmark = pytest.mark.gpu

LIGHT = (abi.PASS_DIFFUSE_DIRECT, abi.PASS_DIFFUSE_INDIRECT, abi.PASS_GLOSSY_DIRECT, abi.PASS_TRANSMISSION_INDIRECT,
         abi.PASS_VOLUME_DIRECT, abi.PASS_EMISSION, abi.PASS_ENVIRONMENT, abi.PASS_GLOSSY_COLOR)
LIGHT_SLOT = dict(zip(LIGHT, (0, 1, 2, 5, 6, 8, 9, 10)))


def even_division(n, d):
    """Cycles' safe_divide_even_color on (..., 3) float32 arrays."""
    with np.errstate(divide="ignore", invalid="ignore"):
        q = np.where(d != 0, n / d, np.float32(0))
    zero = d == 0
    out = q.copy()
    for c in range(3):
        a, b = (c + 1) % 3, (c + 2) % 3
        lo, hi = min(a, b), max(a, b)
        both = np.float32(0.5) * (q[..., lo] + q[..., hi])
        fill = np.where(zero[..., a], q[..., b], np.where(zero[..., b], q[..., a], both))
        out[..., c] = np.where(zero[..., c], fill, q[..., c])
    return out


def expected(kind, film, light, exposure):
    combined, normal, albedo, counts = film
    f = np.float32
    den = np.maximum(counts, 1).astype(np.float32)[..., None]
    if kind == abi.PASS_COMBINED:
        alpha = np.clip(f(1) - combined[..., 3:] / den, f(0), f(1))
        return np.concatenate([combined[..., :3] * (f(exposure) / den), alpha], -1)
    if kind == abi.PASS_NORMAL:
        return normal / den
    if kind == abi.PASS_ALBEDO:
        return albedo / den
    if kind == abi.PASS_SAMPLE_COUNT:
        return np.repeat(counts.astype(np.float32)[..., None], 4, -1)
    slot = LIGHT_SLOT[kind]
    v = light[..., slot, :]
    if slot == 10:
        return v / den
    if slot in (0, 1, 2, 5):
        color = albedo if slot < 2 else light[..., 10 if slot == 2 else 11, :]
        q = even_division(v[..., :3], color[..., :3]) * f(exposure)
        return np.concatenate([q, np.ones_like(q[..., :1])], -1)
    return v * (f(exposure) / den)


@pytest.mark.parametrize("channels", [1, 2, 3, 4])
@pytest.mark.parametrize("width,height", [(1, 1), (17, 15), (64, 4), (257, 1), (96, 61)])
def test_pass_pixels(width, height, channels):
    print(f"case: passes {width}x{height}, {channels} channels", flush=True)
    film_kinds = (abi.PASS_COMBINED, abi.PASS_NORMAL, abi.PASS_ALBEDO, abi.PASS_SAMPLE_COUNT)
    for kinds in (film_kinds, film_kinds + LIGHT):
        s, keep = with_passes(scenes.cornell_settings(width, height), tuple((k, channels) for k in kinds))
        s.integrator.film_exposure = 1.7
        backend = RendererBackend(0, integrator=abi.INTEGRATOR_WAVEFRONT)
        scene = backend.compile_scene(scenes.cornell_lamps()).scene
        session = backend.create_session(scene, s)
        for first, total in ((0, 5), (3, 5)):  # the second call adds to the film
            sink = MemoryOutputSink()
            assert session.render_samples(SampleRange(first, 3 if first == 0 else 2, 0, total), sink)
            film = session.read_film()
            light = session.read_light_passes() if len(kinds) > 4 else None
            for kind in kinds:
                want = expected(kind, film, light, s.integrator.film_exposure)[..., :channels]
                assert np.ascontiguousarray(want, np.float32).tobytes() == sink.passes[kind].tobytes(), kind
        session.close()
        scene.close()
        backend.close()


@pytest.mark.parametrize("total", [1, 257, 1024, 1025, 2049, 8192])
def test_sampler_tables(total):
    """One table per size from 256 to 8192, in one session that is reset."""
    print(f"case: sampler table for {total} samples", flush=True)
    backend = RendererBackend(0)
    scene = backend.compile_scene(scenes.cornell_box()).scene
    s = scenes.cornell_settings(40, 24)
    session = backend.create_session(scene, s)
    for n in (16, total, 16):
        for sample in (0, n // 2, n - 1):
            assert np.array_equal(session.sampler_probe(sample, n, 0, 20), ob.sampler_probe(s, sample, n, 0, 20))
        session.reset(s)
    session.close()
    scene.close()
    backend.close()


def test_concurrent_downloads():
    """Six sessions of one backend read their passes at once, more than the
    stagings that the backend keeps: every sink gets its own film's pixels."""
    print("case: six sessions read their passes at once", flush=True)
    kinds = ((abi.PASS_COMBINED, 4), (abi.PASS_NORMAL, 3), (abi.PASS_ALBEDO, 3), (abi.PASS_SAMPLE_COUNT, 1))
    backend = RendererBackend(0, integrator=abi.INTEGRATOR_WAVEFRONT, graphs=False)
    scene = backend.compile_scene(scenes.cornell_lamps()).scene

    def render(seed):
        s, keep = with_passes(scenes.cornell_settings(200 + 37 * seed, 150), kinds)
        s.seed = seed
        session = backend.create_session(scene, s)
        out = []
        for _ in range(4):
            sink = MemoryOutputSink()
            session.reset(s)
            assert session.render_samples(SampleRange(0, 2, 0, 16), sink)
            out.append({k: v.tobytes() for k, v in sink.passes.items()})
        session.close()
        return out

    alone = [render(seed)[0] for seed in range(6)]
    with ThreadPoolExecutor(6) as pool:
        together = list(pool.map(render, range(6)))
    for want, got in zip(alone, together):
        assert all(g == want for g in got)
    scene.close()
    backend.close()
