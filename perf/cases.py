"""The work that programs on this renderer have it do, as timed cases.

A case is a dict of plain values: `kind` says which public entry points it
takes ("render": RenderSession.render_samples into a sink; "server":
RenderServer requests; "queries": batched ray queries through the C ABI), and
the other keys size it.  `listed()` holds the cases that stand for real use,
`draw()` gives more of the same ranges.  Scenes, resolutions, sample counts
and integrator settings are those of this repository's workloads
(psycles_amd/scenes.py, psycles_amd/serving.py).
"""
from __future__ import annotations

import ctypes as C
import functools
import math
from dataclasses import replace

import numpy as np
import torch

from psycles_amd import abi, scenes, serving
from psycles_amd.render import MemoryOutputSink, RendererBackend, SampleRange, with_passes
from psycles_amd.server import RenderServer

FILM_PASSES = ((abi.PASS_COMBINED, 4), (abi.PASS_NORMAL, 3), (abi.PASS_ALBEDO, 3), (abi.PASS_SAMPLE_COUNT, 1))
LIGHT_PASSES = FILM_PASSES + (
    (abi.PASS_DIFFUSE_DIRECT, 3), (abi.PASS_DIFFUSE_INDIRECT, 3), (abi.PASS_EMISSION, 3), (abi.PASS_ENVIRONMENT, 3))
PASS_NAMES = {abi.PASS_COMBINED: "combined", abi.PASS_NORMAL: "normal", abi.PASS_ALBEDO: "albedo",
              abi.PASS_SAMPLE_COUNT: "sample_count", abi.PASS_DIFFUSE_DIRECT: "diffuse_direct",
              abi.PASS_DIFFUSE_INDIRECT: "diffuse_indirect", abi.PASS_EMISSION: "emission",
              abi.PASS_ENVIRONMENT: "environment"}
FILTERS = {"box": abi.FILTER_BOX, "gaussian": abi.FILTER_GAUSSIAN, "blackman_harris": abi.FILTER_BLACKMAN_HARRIS}
FULL = 224          # mesh frequency of the full-size icosphere: 20 * 224^2 = 1,003,520 triangles
QUERY_FAR = 1000.0  # far end of the closest-hit queries; misses report it as their distance

# Per scene: rays per camera sample, binary-SAH node visits (two box tests of
# 12 operations each) and triangle tests (45 operations) per ray, as counted
# on the workloads' frames.
COUNTS = {"cornell": (5.9, 11.2, 7.3), "lamps": (6.5, 11.2, 7.3), "instanced": (2.06, 46.8, 8.6),
          "many_lights": (4.86, 94.8, 15.1), "slabs": (15.7, 12.0, 9.0)}
# Relative cost of one camera sample, from the frames' times; bounds a drawn case.
COST = {"cornell": 0.35, "lamps": 0.6, "instanced": 0.19, "many_lights": 1.0, "slabs": 0.8}


def render_case(name, scene, width, height, spp, **more):
    case = {"name": name, "kind": "render", "scene": scene, "detail": FULL, "count": 64, "width": width,
            "height": height, "spp": spp, "calls": 1, "batch": spp, "integrator": "wavefront", "generated": True,
            "light_passes": False, "filter": "box"}
    case.update(more)
    return case


def listed():
    return [
        # an interactive viewport on a small scene, refined one sample per
        # call and shown after each: latency, launches and readback
        render_case("viewport_cornell", "cornell", 256, 256, 4, calls=4, batch=1, generated=False),
        # the Cornell box as a whole frame
        render_case("frame_cornell", "cornell", 640, 400, 16),
        # a backend with its default options: one lane per path
        render_case("default_cornell", "cornell", 640, 400, 4, integrator="default", generated=False),
        # a viewport on the 1M-triangle, 64-instance scene
        render_case("viewport_instanced", "instanced", 640, 400, 4, batch=4, generated=False),
        # the headline frame
        render_case("frame_instanced", "instanced", 1920, 1080, 64),
        # the smallest request on the heaviest scene: one sample through the light tree
        render_case("viewport_many_lights", "many_lights", 256, 256, 1, generated=False),
        # the many-light frame
        render_case("frame_many_lights", "many_lights", 1920, 1080, 32),
        # long paths through stacked transparent slabs, ragged size
        render_case("uneven_slabs", "slabs", 773, 773, 37, count=13),
        # a frame with light passes for compositing, odd window, wide filter
        render_case("light_passes", "lamps", 427, 311, 8, light_passes=True, filter="blackman_harris"),
        # requests of mixed size with parameter edits between them, all at
        # once, on a server with resident scenes
        {"name": "server_mixed", "kind": "server", "requests": 12, "detail": 64, "count": 16, "largest": 1280 * 720,
         "samples": 16, "mix": 4},
        # ray queries of a host program: a small batch from host memory
        {"name": "queries_host", "kind": "queries", "scene": "instanced", "detail": 8, "count": 15, "rays": 4096,
         "host": True, "shadow": 0.5},
        # a large batch resident on the device, against the full-size scene
        {"name": "queries_device", "kind": "queries", "scene": "instanced", "detail": FULL, "count": 64,
         "rays": 1 << 21, "host": False, "shadow": 0.5},
    ]


def log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def draw(rng):
    kind = rng.choice(("render", "render", "render", "render", "queries", "server"))
    if kind == "server":
        return {"kind": kind, "requests": rng.randint(3, 14), "detail": int(log_uniform(rng, 16, 96)),
                "count": rng.randint(4, 32), "largest": int(log_uniform(rng, 256 * 256, 1280 * 720)),
                "samples": rng.choice((1, 4, 16)), "mix": rng.randint(0, 1 << 16)}
    if kind == "queries":
        scene = rng.choice(("cornell", "instanced", "slabs"))
        return {"kind": kind, "scene": scene, "detail": int(log_uniform(rng, 8, FULL)), "count": rng.randint(3, 64),
                "rays": int(log_uniform(rng, 500, 1 << 21)), "host": rng.random() < 0.5,
                "shadow": round(rng.random(), 2)}
    scene = rng.choice(tuple(COST))
    default = rng.random() < 0.2
    width, height = int(log_uniform(rng, 100, 1920)), int(log_uniform(rng, 70, 1080))
    passes = not default and rng.random() < 0.15
    budget = 0.5 * COST["many_lights"] * 1920 * 1080 * 32 / (COST[scene] * (8 if default else 1))
    most = max(1, min(64, int(budget / (width * height))))
    spp = max(1, int(log_uniform(rng, 1, most)))
    case = render_case("", scene, width, height, spp, detail=int(log_uniform(rng, 16, FULL)),
                       count=rng.randint(8, 64) if scene in ("instanced", "many_lights") else rng.randint(1, 16),
                       batch=spp if rng.random() < 0.6 else rng.randint(1, spp), light_passes=passes,
                       integrator="default" if default else "wavefront",
                       generated=not default and rng.random() < 0.5, filter=rng.choice(tuple(FILTERS)))
    case["calls"] = 1 if spp == 1 or rng.random() < 0.7 else 2
    del case["name"]
    return case


# ---- what a program has in hand -------------------------------------------

@functools.lru_cache(maxsize=4)
def geometry(scene, detail, count):
    """The scene as a program reads it from its files."""
    if scene == "cornell":
        return scenes.cornell_box()
    if scene == "lamps":
        return scenes.cornell_lamps()
    if scene == "instanced":
        return scenes.instanced_icospheres(frequency=detail, instances=count)
    if scene == "many_lights":
        return scenes.many_lights(frequency=detail, instances=count, emissive=10000 * count // 64,
                                  points=4 * count, spots=count)
    rng = np.random.RandomState(count)
    return scenes.uneven_slabs(list(0.5 + 0.45 * rng.rand(count)),
                               [tuple(0.2 + 0.7 * rng.rand(3)) for _ in range(3 + count)],
                               [(-1.5 + 3.0 * rng.rand(), -2.5 + 1.5 * rng.rand(), 90.0 * rng.rand())
                                for _ in range(3)])


def edited(material, factor):
    return replace(material, parameters=serving.edited_parameters(material.instructions, material.parameters, factor))


def variant(scene, detail, count, seed):
    """The scene with the material values and the camera place of one job."""
    snap = geometry(scene, detail, count)
    rng = np.random.RandomState(seed % (1 << 31))
    move = np.eye(4, dtype=np.float32)
    reach = 1.0 if scene in ("instanced", "many_lights") else 0.05
    move[:3, 3] = reach * (2.0 * rng.rand(3) - 1.0)
    camera = replace(snap.camera, transform=(move @ snap.camera.transform).astype(np.float32))
    return replace(snap, materials=[edited(m, 0.9 + 0.2 * rng.rand()) for m in snap.materials], camera=camera)


@functools.lru_cache(maxsize=None)
def backend(integrator, batch, generated):
    """One backend per process and option set."""
    if integrator == "default":
        return RendererBackend(0)
    return RendererBackend(0, integrator=abi.INTEGRATOR_WAVEFRONT, max_samples_per_dispatch=batch,
                           generated_programs=generated)


def compiled(be, snap):
    comp = be.compile_scene(snap)
    if not comp.ok():
        raise RuntimeError("; ".join(d.message for d in comp.diagnostics))
    return comp.scene


def scene_settings(scene, width, height):
    if scene in ("cornell", "lamps"):
        return scenes.cornell_settings(width, height)
    if scene == "slabs":
        return scenes.uneven_settings(width, 0)
    return serving.scene_settings(scene, width, height)


def settings_of(case, seed):
    s = scene_settings(case["scene"], case["width"], case["height"])
    s.width, s.height = case["width"], case["height"]
    s.window_width, s.window_height = case["width"], case["height"]
    s.seed = seed % (1 << 31)
    if case["filter"] != "box":
        s.pixel_filter, s.filter_width = FILTERS[case["filter"]], 1.5
    return with_passes(s, LIGHT_PASSES if case["light_passes"] else FILM_PASSES)


def prepare(case, seed):
    if case["kind"] == "queries":
        return prepare_queries(case, seed)
    if case["kind"] == "server":
        return prepare_server(case, seed)
    be = backend(case["integrator"], case["batch"], case["generated"])
    scene = compiled(be, variant(case["scene"], case["detail"], case["count"], seed))
    settings, keep = settings_of(case, seed)
    session = be.create_session(scene, settings)
    return {"case": case, "session": session, "settings": settings, "keep": keep}


def prepare_server(case, seed):
    """Resident scenes, a server, and a list of submissions: renders drawn as
    the serving stream draws them, 30 % of the steps parameter edits."""
    be = backend("wavefront", 4, False)
    names = ("cornell", "instanced", "lamps")
    snaps = {n: variant(n, case["detail"], case["count"], seed) for n in names}
    resident = {n: compiled(be, s) for n, s in snaps.items()}
    rng = np.random.RandomState(case["mix"])
    steps, first = [], {}
    sizes = [r for r in serving.RESOLUTIONS if r[0] * r[1] <= case["largest"]] or [serving.RESOLUTIONS[0]]
    while sum(s[0] == "render" for s in steps) < case["requests"]:
        name = names[rng.randint(len(names))]
        if rng.rand() < 0.3:
            at = rng.randint(len(snaps[name].materials))
            material = snaps[name].materials[at]
            first.setdefault((name, at), material.parameters)
            steps.append(("edit", name, at, edited(material, 0.8 + 0.4 * rng.rand()).parameters))
            continue
        w, h = sizes[rng.randint(len(sizes))]
        if rng.rand() < 0.3:
            w, h = w - rng.randint(1, 64), h - rng.randint(1, 48)
        s = scene_settings(name, w, h)
        s.seed = (seed + len(steps)) % (1 << 31)
        spp = [n for n in serving.SAMPLE_COUNTS if n <= case["samples"]]
        steps.append(("render", name, s, spp[rng.randint(len(spp))]))
    # a pass starts from the materials as they were loaded
    steps = [("edit", name, at, p) for (name, at), p in first.items()] + steps
    return {"case": case, "server": RenderServer(be), "resident": resident, "steps": steps}


def query_records(case, seed):
    """Query records between random points of the scene's box: closest hits
    along unbounded rays, and shadow segments."""
    n = case["rays"]
    rng = np.random.RandomState(seed % (1 << 31))
    center, reach = ((0.0, -1.0, 0.0), 26.0) if case["scene"] == "instanced" else ((0.0, 0.0, 0.5), 1.9)
    a = np.asarray(center) + reach * (2.0 * rng.rand(n, 3) - 1.0)
    b = np.asarray(center) + reach * (2.0 * rng.rand(n, 3) - 1.0)
    shadow = rng.rand(n) < case["shadow"]
    along = b - a
    length = np.linalg.norm(along, axis=1)
    q = np.zeros((n, 16), dtype=np.float32)
    words = q.view(np.uint32)
    q[:, 0:3] = a
    q[:, 4:7] = along / length[:, None]
    q[:, 7] = np.where(shadow, length, QUERY_FAR)
    words[:, 8] = np.where(shadow, abi.VIS_SHADOW, abi.VIS_ALL)
    words[:, 9:13] = abi.INVALID_ID
    words[:, 13] = np.where(shadow, abi.QUERY_SHADOW, abi.QUERY_CLOSEST)
    words[:, 15] = 8
    return q


def prepare_queries(case, seed):
    be = backend("wavefront", 4, False)
    scene = compiled(be, variant(case["scene"], case["detail"], case["count"], seed))
    q = query_records(case, seed)
    state = {"case": case, "scene": scene, "lib": be.lib, "host": q}
    if case["host"]:
        state["hits"] = np.zeros((len(q), 12), dtype=np.float32)
    else:
        state["queries"] = torch.from_numpy(q).cuda()
        state["hits"] = torch.zeros((len(q), 12), dtype=torch.float32, device="cuda")
    return state


# ---- one pass --------------------------------------------------------------

def run(state):
    case = state["case"]
    if case["kind"] == "queries":
        return run_queries(state)
    if case["kind"] == "server":
        return run_server(state)
    session, spp, calls = state["session"], case["spp"], case["calls"]
    session.reset(state["settings"])
    out, first = [], 0
    for c in range(calls):
        count = spp * (c + 1) // calls - first
        sink = MemoryOutputSink()
        if not session.render_samples(SampleRange(first, count, 0, spp), sink):
            raise RuntimeError(f"render_samples returned false ({session.last_status})")
        first += count
        out.append({PASS_NAMES[k]: v for k, v in sink.passes.items()})
    return out


def run_server(state):
    server, resident = state["server"], state["resident"]
    requests = []
    for step in state["steps"]:
        if step[0] == "edit":
            server.update_parameters(resident[step[1]], step[2], step[3])
        else:
            requests.append(server.submit(resident[step[1]], step[2], 0, step[3], step[3]))
    films = []
    for r in requests:
        if not r.wait():
            raise RuntimeError("a request was not completed")
        films.append(r.read_film())
        r.release()
    return films


def run_queries(state):
    lib, scene, n = state["lib"], state["scene"], state["case"]["rays"]
    hits = state["hits"]
    if state["case"]["host"]:
        abi.check("psx_scene_intersect", lib.psx_scene_intersect(
            scene.handle, state["host"].ctypes.data_as(C.POINTER(abi.RayQuery)), n,
            hits.ctypes.data_as(C.POINTER(abi.RayHit))))
        words = hits.view(np.int32)
    else:
        abi.check("psx_scene_intersect_device", lib.psx_scene_intersect_device(
            scene.handle, state["queries"].data_ptr(), n, hits.data_ptr()))
        words = hits.view(torch.int32)
    return {"distance": hits[:, 0], "uv": hits[:, 1:3], "identity": words[:, 3:6], "transmittance": hits[:, 8:11]}


# ---- what it takes, and what it should give ---------------------------------

def triangles(scene, detail, count):
    return {"cornell": 34, "lamps": 34, "slabs": 2 * count + 38, "instanced": 20 * detail * detail + 2,
            "many_lights": 20 * detail * detail + 2 + 10000 * count // 64}[scene]


def ray_flops(scene):
    _, nodes, tris = COUNTS[scene]
    return 24.0 * nodes + 45.0 * tris


def work(case):
    if case["kind"] == "queries":
        return {"bytes": 112.0 * case["rays"] + 36.0 * triangles(case["scene"], case["detail"], case["count"]),
                "flops": case["rays"] * ray_flops(case["scene"])}
    if case["kind"] == "server":
        pixels, samples = case["largest"] / 2.0, case["samples"] / 2.0
        return {"bytes": case["requests"] * pixels * 52.0 + 36.0 * triangles("instanced", case["detail"], 1),
                "flops": case["requests"] * pixels * samples * COUNTS["cornell"][0] * ray_flops("cornell")}
    channels = sum(c for _, c in (LIGHT_PASSES if case["light_passes"] else FILM_PASSES))
    pixels = case["width"] * case["height"]
    rays = pixels * case["spp"] * COUNTS[case["scene"]][0]
    return {"bytes": 4.0 * channels * pixels * case["calls"]
            + 36.0 * triangles(case["scene"], case["detail"], case["count"]),
            "flops": rays * ray_flops(case["scene"])}


def tolerance(case):
    """Four times what two implementations at the same precision differ by:
    the films against the CPU renderer of tests/ (at most 9.4e-6 in the 2-norm
    and 7.1e-4 at a value, on the Cornell box), the queries against 64 bits
    (2.6e-5, of the barycentrics)."""
    if case["kind"] == "queries":
        return {"rel": 1e-4, "max": 2e-2, "differ": 1e-5}
    return {"rel": 4e-5, "max": 4e-3, "differ": 0.0}


def shadow_factor(material):
    """What a shadow ray keeps through a surface of `material`: the share of
    the transparent side of a mix, nothing through the other closures."""
    op, _, b, factor = material.instructions[material.root][:4]
    if op == abi.CLOSURE_MIX and material.instructions[b][0] == abi.CLOSURE_TRANSPARENT:
        return float(material.parameters[factor])
    return 0.0


def exact_queries(case, seed):
    """Every query against every triangle in 64 bits (Moeller and Trumbore)."""
    device = "cuda" if torch.cuda.is_available() else "cpu"
    snap = variant(case["scene"], case["detail"], case["count"], seed)
    corners, factor = [], []
    for inst in snap.instances:
        mesh = snap.meshes[inst.mesh]
        m = torch.as_tensor(np.asarray(inst.transform), dtype=torch.float64, device=device)
        p = torch.as_tensor(mesh.positions, dtype=torch.float64, device=device) @ m[:3, :3].T + m[:3, 3]
        corners.append(p[torch.as_tensor(mesh.triangles.astype(np.int64), device=device)])
        slots = inst.material_overrides or mesh.material_slots
        which = (mesh.triangle_material_slots if mesh.triangle_material_slots is not None
                 else np.zeros(len(mesh.triangles), dtype=np.int64))
        factor.append(torch.tensor([shadow_factor(snap.materials[slots[min(int(w), len(slots) - 1)]]) for w in which],
                                   dtype=torch.float64, device=device))
    p, keep = torch.cat(corners), torch.cat(factor)
    e1, e2 = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    rays = torch.as_tensor(query_records(case, seed), device=device)
    shadow = rays[:, 13].contiguous().view(torch.int32) == abi.QUERY_SHADOW
    rays = rays.double()
    n = case["rays"]
    distance, uv = rays[:, 7].clone(), torch.zeros((n, 2), dtype=torch.float64, device=device)
    through = torch.zeros((n, 3), dtype=torch.float64, device=device)
    step = max(1, 20_000_000 // len(p))
    for at in range(0, n, step):
        o, d, far = rays[at:at + step, None, 0:3], rays[at:at + step, None, 4:7], rays[at:at + step, 7]
        h = torch.linalg.cross(d.expand(-1, len(p), -1), e2[None].expand(len(o), -1, -1))
        inv = 1.0 / (h * e1).sum(-1)
        s = o - p[:, 0]
        u = (s * h).sum(-1) * inv
        g = torch.linalg.cross(s, e1[None].expand(len(o), -1, -1))
        v = (d * g).sum(-1) * inv
        t = (e2 * g).sum(-1) * inv
        hit = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= 0) & (t <= far[:, None])
        t = torch.where(hit, t, torch.inf)
        best = t.argmin(1)
        row = torch.arange(len(o), device=device)
        found = hit.any(1) & ~shadow[at:at + step]
        distance[at:at + step] = torch.where(found, t[row, best], far)
        uv[at:at + step] = torch.where(found[:, None], torch.stack((u[row, best], v[row, best]), 1), 0.0)
        left = torch.where(hit, keep, 1.0).prod(1)
        left = torch.where(hit.sum(1) > 8, 0.0, left)  # transparent_max of the queries
        through[at:at + step] = torch.where(shadow[at:at + step], left, 0.0)[:, None]
    return {"distance": distance, "uv": uv, "identity": None, "transmittance": through}


def exact(case, seed):
    """Ray queries have 64-bit answers; of a film, a Monte Carlo estimate over
    the sampler's own points, only the sample count has one."""
    if case["kind"] == "queries":
        total = triangles(case["scene"], case["detail"], case["count"]) * case["rays"]
        if case["scene"] == "instanced":
            total = (20 * case["detail"] ** 2 * case["count"] + 2) * case["rays"]
        return exact_queries(case, seed) if total <= 2_000_000_000 else None
    if case["kind"] == "server":
        return None
    out = []
    for c in range(case["calls"]):
        names = [PASS_NAMES[k] for k, _ in (LIGHT_PASSES if case["light_passes"] else FILM_PASSES)]
        done = case["spp"] * (c + 1) // case["calls"]
        out.append({n: None for n in names})
        out[-1]["sample_count"] = np.full((case["height"], case["width"], 1), float(done))
    return out
