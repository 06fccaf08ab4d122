"""Performance cases: what users of this renderer have it do, from one pick to a frame of 205 M triangles.

Every case goes through the package's public entry points and ends where a
user's program gets its result: a NumPy image, product arrays, hit arrays,
or a display frame in device memory.  Scenes are the seeded generators of
``ordinarylight_amd.workloads``; sizes come from the benchmark, the tests
and common image formats.

A case is a dict of plain values:

* ``kind``: ``pick``, ``frame``, ``products``, ``display``, ``batch``,
  ``animate``, ``trace`` or ``reference`` (see ``run``);
* ``scene``, ``size``: generator and its size (triangles, or instances);
* ``width``, ``height``, ``samples``, ``bounces``: the image and its paths;
* ``builder``: the hierarchy builder (``lbvh``: the renderer's default,
  rebuilt quickly; ``sah``: for static scenes);
* further options that only some kinds read.
"""

import math

import numpy as np
import torch

from ordinarylight_amd import workloads
from ordinarylight_amd.batch import BatchEngine, EngineSettings, Job
from ordinarylight_amd.renderers.hip import (
    DeviceContext, DeviceScene, HipPathTracer, HipReferenceRenderer, HipRendererConfig,
)


def listed():
    return [
        # A click in a viewport: one primary ray, all latency.
        {"name": "pick", "kind": "pick", "scene": "room", "size": 40_000, "width": 641, "height": 479,
         "samples": 1, "bounces": 1, "builder": "lbvh"},
        # A thumbnail or preview: a few small launches per bounce.
        {"name": "preview_room", "kind": "frame", "scene": "room", "size": 10_000, "width": 256, "height": 256,
         "samples": 1, "bounces": 4, "builder": "lbvh"},
        # An odd-sized still with point and spot lights, per-domain light
        # sampling and Russian roulette.
        {"name": "lights_odd", "kind": "frame", "scene": "terrain_lights", "size": 100_000, "width": 641,
         "height": 479, "samples": 4, "bounces": 8, "builder": "sah", "per_domain": True, "roulette": True},
        # Textured materials, glass and an image environment.
        {"name": "textured", "kind": "frame", "scene": "textured", "size": 40, "width": 640, "height": 360,
         "samples": 4, "bounces": 6, "builder": "lbvh"},
        # Colour with depth, normals, ids and variance, for a denoiser or compositor.
        {"name": "products", "kind": "products", "scene": "room", "size": 160_000, "width": 800, "height": 600,
         "samples": 4, "bounces": 4, "builder": "sah"},
        # An interactive viewer: one sample per pixel of a 1080p frame,
        # tone-mapped into a device buffer.
        {"name": "display_1080p", "kind": "display", "scene": "terrain", "size": 500_000, "width": 1920,
         "height": 1080, "samples": 1, "bounces": 5, "builder": "lbvh"},
        # The benchmark's frame: 1 M triangles, 1080p, 8 samples, 8 bounces.
        {"name": "frame_1080p", "kind": "frame", "scene": "terrain", "size": 1_000_000, "width": 1920,
         "height": 1080, "samples": 8, "bounces": 8, "builder": "sah"},
        # The benchmark's two-level frame: 10,000 instances, 20 % glass,
        # 100,000 emitters through reservoir resampling, 16 bounces.
        {"name": "instanced_1080p", "kind": "frame", "scene": "spheres", "size": 10_000, "width": 1920,
         "height": 1080, "samples": 4, "bounces": 16, "builder": "sah", "restir": 32},
        # A render farm's queue: mixed jobs over resident scenes in one engine.
        {"name": "batch_mixed", "kind": "batch", "scene": "mixed", "size": 250_000, "width": 640, "height": 640,
         "samples": 8, "bounces": 8, "builder": "sah", "jobs": 24},
        # An animated mesh: the resident hierarchy follows the vertices, then a frame.
        {"name": "animate", "kind": "animate", "scene": "terrain", "size": 100_000, "width": 512, "height": 512,
         "samples": 1, "bounces": 4, "builder": "lbvh"},
        # Ray queries from a user's own arrays (visibility, baking).
        {"name": "trace_rays", "kind": "trace", "scene": "terrain", "size": 100_000, "width": 250_001, "height": 1,
         "samples": 1, "bounces": 1, "builder": "sah"},
        # The reference estimator on its own benchmark frame.
        {"name": "reference", "kind": "reference", "scene": "box", "size": 36, "width": 256, "height": 256,
         "samples": 4, "bounces": 4, "builder": "lbvh"},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pick", "frame", "frame", "frame", "products", "display", "batch", "animate", "trace",
                       "reference"])
    case = {"kind": kind, "samples": 1, "bounces": rng.choice([2, 3, 4, 5, 6, 8]),
            "builder": rng.choice(["lbvh", "sah"])}
    if kind == "pick":
        case.update(scene=rng.choice(["room", "terrain"]), size=_log_uniform(rng, 10_000, 500_000),
                    width=_log_uniform(rng, 128, 3840), height=_log_uniform(rng, 128, 2160), bounces=1)
    elif kind == "reference":
        case.update(scene="box", size=36, width=_log_uniform(rng, 32, 320), height=_log_uniform(rng, 32, 320),
                    samples=rng.randint(1, 4), bounces=rng.randint(1, 4))
    elif kind == "trace":
        case.update(scene=rng.choice(["room", "terrain"]), size=_log_uniform(rng, 10_000, 100_000),
                    width=_log_uniform(rng, 100, 250_000), height=1, bounces=1)
    elif kind == "batch":
        case.update(scene="mixed", size=_log_uniform(rng, 20_000, 250_000), width=rng.randint(200, 640),
                    height=rng.randint(200, 640), samples=8, bounces=8, jobs=rng.randint(4, 24))
    elif kind == "animate":
        case.update(scene=rng.choice(["room", "terrain"]), size=_log_uniform(rng, 10_000, 100_000),
                    width=rng.randint(128, 640), height=rng.randint(128, 512), builder="lbvh")
    else:
        scene = rng.choice(["room", "terrain", "terrain_lights", "textured", "spheres"])
        if kind == "products":
            scene = rng.choice(["room", "terrain"])
        case.update(scene=scene, width=_log_uniform(rng, 97, 1920), height=_log_uniform(rng, 65, 1080),
                    samples=rng.choice([1, 1, 2, 4, 8]))
        if scene == "textured":
            case.update(size=40)
        elif scene == "spheres":
            case.update(size=_log_uniform(rng, 50, 4000), samples=min(case["samples"], 4),
                        restir=rng.choice([0, 1, 8, 32]))
        else:
            case.update(size=_log_uniform(rng, 10_000, 500_000))
        if scene == "terrain_lights":
            case.update(per_domain=rng.random() < 0.5, roulette=rng.random() < 0.5)
        if kind == "display":
            # NV12 and P010 need a width divisible by 4 and an even height.
            case.update(width=4 * max(case["width"] // 4, 16), height=2 * max(case["height"] // 2, 16),
                        format=rng.choice(["rgba8", "nv12", "p010"]))
    return case


# ---- inputs -----------------------------------------------------------------------------------
def _terrain(seed, triangles):
    k = max(4, int(round(math.sqrt(triangles / 4.0))))
    return workloads.terrain(seed, nx=2 * k + 1, nz=k + 1, chunk=max(50, k // 4), emissive_quads=32)


def _scene(name, size, seed):
    if name == "box":
        return workloads.box_room(seed)
    if name == "room":
        return workloads.tessellated_room(seed, size)
    if name == "textured":
        return workloads.textured_room(seed, open_sky=True)
    if name == "spheres":
        return workloads.instanced_spheres(seed, instances=size, emitters=10 * size)
    scene, camera = _terrain(seed, size)
    if name == "terrain_lights":
        span = np.asarray(camera.target, np.float64)
        scene.add_point_light(tuple(span + (0.0, 60.0, 0.0)), color=(1.0, 0.8, 0.6), intensity=4000.0)
        scene.add_spot_light(tuple(span + (20.0, 80.0, -30.0)), (0.0, -1.0, 0.2), intensity=8000.0,
                             inner_cone_angle=0.4, outer_cone_angle=0.8)
    return scene, camera


def _config(case):
    options = {}
    if case.get("per_domain"):
        options.update(wavefront_unified_secondary_nee=False, area_light_samples=2)
    if case.get("roulette"):
        options.update(wavefront_russian_roulette=True)
    if case.get("restir"):
        options.update(wavefront_restir_di=True, wavefront_restir_candidates=case["restir"],
                       wavefront_restir_spatial_reuse=True, wavefront_restir_spatial_neighbors=1)
    return HipRendererConfig(max_bounces=case["bounces"], samples_per_pixel=case["samples"],
                             bvh_builder=case["builder"], **options)


def _rays(vertices, count, seed):
    """Origins round the scene's box, directions towards points inside it and
    (every second ray) points close to its surface, and a range that covers
    the scene."""
    rng = np.random.default_rng(seed)
    lo, hi = vertices.min(0).astype(np.float64), vertices.max(0).astype(np.float64)
    pad = 0.2 * (hi - lo)
    o = rng.uniform(lo - pad, hi + pad, (count, 3))
    target = rng.uniform(lo, hi, (count, 3))
    near = vertices[rng.integers(0, len(vertices), len(target[1::2]))]
    target[1::2] = near + rng.normal(0.0, 0.002 * np.linalg.norm(hi - lo), near.shape)
    o, target = o.astype(np.float32), target.astype(np.float32)
    d = target - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return o, d, float(4.0 * np.linalg.norm(hi - lo))


def _pick_pixel(case, seed):
    """A seeded position in the lower half of the viewport, where the scenes have surfaces."""
    rng = np.random.default_rng(seed)
    return (float(rng.uniform(0.1, 0.9) * case["width"]), float(rng.uniform(0.5, 0.95) * case["height"]))


class State:
    """What the user's program holds between passes; frees the device side with itself."""

    def __init__(self):
        self.owned = []

    def own(self, thing):
        self.owned.append(thing)
        return thing

    def __del__(self):
        for thing in reversed(self.owned):
            thing.close()


def prepare(case, seed):
    st = State()
    st.case = dict(case)
    kind = case["kind"]
    st.frame_index = seed % 1024
    if kind == "batch":
        # Four resident scenes and a seeded job list over them.
        ctx = st.own(DeviceContext(0))
        scenes = {}
        for k, (name, size) in enumerate((("room", case["size"] // 4), ("terrain", case["size"] // 2),
                                          ("room", case["size"] // 16 + 100), ("terrain", case["size"]))):
            scene, camera = _scene(name, size, seed + k)
            scenes[k] = (st.own(DeviceScene(ctx, scene, 2, builder=case["builder"])), camera)
        # (The list belongs to the case, the scenes and frames to the seed.)
        rng = np.random.default_rng(case["jobs"])
        edge = max(case["width"], case["height"])
        st.jobs = []
        for j in range(case["jobs"]):
            device_scene, camera = scenes[int(rng.integers(4))]
            w, h = (int(round(math.exp(rng.uniform(math.log(min(96, edge - 1)), math.log(edge))))) for _ in range(2))
            st.jobs.append(Job(device_scene, camera, w, h, int(rng.choice((1, 2, 4, case["samples"]))),
                               st.frame_index + j,
                               max_bounces=int(rng.choice((4, case["bounces"])))))
        st.engine = st.own(BatchEngine(ctx, EngineSettings(path_slots=1 << 24)))
        return st
    scene, camera = _scene(case["scene"], case["size"], seed)
    st.scene, st.camera = scene, camera
    if kind == "trace":
        ctx = st.own(DeviceContext(0))
        st.device_scene = st.own(DeviceScene(ctx, scene, 2, builder=case["builder"]))
        st.origins, st.directions, st.tmax = _rays(st.device_scene.packed.positions, case["width"], seed)
        return st
    if kind == "reference":
        st.renderer = st.own(HipReferenceRenderer(samples_per_pixel=case["samples"], max_bounces=case["bounces"],
                                                  seed=seed))
        st.renderer.replace_scene(scene)
        return st
    st.renderer = st.own(HipPathTracer(_config(case)))
    st.renderer.replace_scene(scene)
    if kind == "pick":
        st.pixel = _pick_pixel(case, seed)
    elif kind == "display":
        st.format = case.get("format", "rgba8")
        w, h = case["width"], case["height"]
        shape, dtype = {"rgba8": ((h, w, 4), torch.uint8), "nv12": ((h * 3 // 2, w), torch.uint8),
                        "p010": ((h * 3 // 2, w), torch.int16)}[st.format]
        st.out = torch.zeros(shape, dtype=dtype, device="cuda")
        torch.cuda.synchronize()
    elif kind == "animate":
        st.resource = scene.mesh_resources[0]
        rest = st.resource.vertices
        rng = np.random.default_rng(seed)
        extent = float(np.ptp(rest, axis=0).max())
        st.poses = [(rest + (0.01 * extent * np.sin(rest * rng.uniform(3.0, 9.0) / extent
                                                    + rng.uniform(0, 6.0)))).astype(np.float32) for _ in range(2)]
    return st


# ---- one pass ---------------------------------------------------------------------------------
def run(state):
    case = state.case
    kind, w, h = case["kind"], case["width"], case["height"]
    if kind == "frame":
        return state.renderer.render_frame(state.scene, state.camera, w, h, frame_index=state.frame_index)
    if kind == "products":
        return state.renderer.render_products(
            state.scene, state.camera, w, h, frame_index=state.frame_index,
            outputs=("color", "variance", "depth", "normal", "object_id", "material_id"))
    if kind == "display":
        state.renderer.render_output(state.scene, state.camera, w, h, pixel_format=state.format,
                                     frame_index=state.frame_index, device_out=state.out.data_ptr())
        return state.out
    if kind == "pick":
        hit = state.renderer.pick(state.scene, state.camera, (w, h), state.pixel)
        if hit is None:
            return {"object": 0, "triangle": -1, "distance": 0.0, "position": np.zeros(3), "weights": np.zeros(3)}
        return {"object": hit.object_id, "triangle": hit.primitive_index, "distance": hit.distance,
                "position": np.asarray(hit.position), "weights": np.asarray(hit.barycentric)}
    if kind == "batch":
        ids = [state.engine.submit(job) for job in state.jobs]
        state.engine.run()
        return [state.engine.result(i)[0] for i in ids]
    if kind == "animate":
        frames = []
        for pose in state.poses:
            state.scene.update_mesh_resource(state.resource, vertices=pose)
            frames.append(state.renderer.render_frame(state.scene, state.camera, w, h,
                                                      frame_index=state.frame_index))
        return frames
    if kind == "trace":
        t, u, v, triangle = state.device_scene.trace(state.origins, state.directions, 0.001, state.tmax)
        return {"t": t, "u": u, "v": v, "triangle": triangle}
    return state.renderer.render_frame(state.scene, state.camera, w, h, frame_index=state.frame_index)


# ---- what a pass cannot do without ------------------------------------------------------------
def work(case):
    """Scene read once and results written once; for every ray a descent of a
    balanced hierarchy (a box test per level and side) and two triangle tests,
    for every surface hit its shading.  Paths live about two segments, and
    every second hit sends a shadow ray."""
    kind = case["kind"]
    triangles = {"spheres": 5 * 20_480 + 10 * case["size"], "mixed": 2 * case["size"]}.get(case["scene"], case["size"])
    pixels = case["width"] * case["height"]
    paths, out = pixels * case["samples"], 16 * pixels
    if kind == "pick":
        paths, out = 1, 48
    elif kind == "trace":
        paths, out = case["width"], 48 * case["width"]
    elif kind == "batch":
        # Mean area and samples of the job list.
        edge = max(case["width"], case["height"])
        mean = ((edge - 95) / math.log(edge / 95.0)) ** 2
        paths, out = int(case["jobs"] * mean * 3.75), int(case["jobs"] * mean * 16)
    elif kind == "products":
        out = 44 * pixels
    elif kind == "display":
        out = {"rgba8": 4.0, "nv12": 1.5, "p010": 3.0}[case.get("format", "rgba8")] * pixels
    elif kind == "animate":
        paths, out = 2 * paths, 2 * out + 2 * 16 * triangles
    rays = paths * (1.0 if kind in ("pick", "trace") else 3.0)
    per_ray = 2.0 * math.log2(triangles + 1.0) * 15.0 + 2.0 * 50.0
    shading = 0.0 if kind in ("pick", "trace") else 300.0 * 2.0 * paths
    touched = min(96.0 * triangles, rays * 48.0 * 2.0)
    return {"bytes": float(out + touched), "flops": rays * per_ray + shading}


def tolerance(case):
    """Float32 arithmetic in another order: the C restatement of the estimator
    (same sample streams, same closest hits, its own order of traversal and
    operations) differs from these images by 1e-8 to 1.4e-6, most with
    textures; ray distances differ from 64-bit ones by 1e-7 except where a ray
    grazes an edge.  Ids and display bytes are whole values and stay the same."""
    if case["kind"] == "display":
        return "exact"
    return {"rel": 6e-6}


# ---- 64-bit results ---------------------------------------------------------------------------
def _closest(origins, directions, corners, tmin, tmax):
    """Closest hits of float64 rays over all triangles by brute force: t, u, v, triangle (-1: none)."""
    v0, e1, e2 = corners[:, 0], corners[:, 1] - corners[:, 0], corners[:, 2] - corners[:, 0]
    parts = []
    step = max(1, int(1e8 // len(corners)))
    for first in range(0, len(origins), step):
        o, d = origins[first:first + step, None, :], directions[first:first + step, None, :]
        p = torch.linalg.cross(d, e2[None].expand(d.shape[0], -1, -1))
        det = (e1[None] * p).sum(-1)
        inv = 1.0 / torch.where(det == 0.0, torch.ones_like(det), det)
        s = o - v0[None]
        u = (s * p).sum(-1) * inv
        del p
        q = torch.linalg.cross(s, e1[None].expand(s.shape[0], -1, -1))
        v = (d * q).sum(-1) * inv
        t = (e2[None] * q).sum(-1) * inv
        inside = (det != 0.0) & (u >= 0.0) & (v >= 0.0) & (u + v <= 1.0) & (t >= tmin) & (t <= tmax)
        best, at = torch.where(inside, t, torch.full_like(t, float("inf"))).min(1)
        row = torch.arange(len(at), device=at.device)
        hit = torch.isfinite(best)
        zero = torch.zeros_like(best)
        parts.append(torch.stack((torch.where(hit, best, zero + tmax), torch.where(hit, u[row, at], zero),
                                  torch.where(hit, v[row, at], zero), torch.where(hit, at.double(), zero - 1.0)), 1))
    return torch.cat(parts).cpu().numpy()


def _hash(v):
    for shift, factor in ((16, 2146121005), (15, 2221713035)):
        v = ((v ^ (v >> shift)) * factor) & 0xFFFFFFFF
    return v ^ (v >> 16)


def _pixel_ray(camera, width, height, x, y):
    """The hash-jittered camera ray of (pixel, frame 0, sample 0) in 64 bits."""
    state = _hash(_hash((y * width + x) ^ _hash(0) ^ _hash(1)))
    jx, state = state / 2.0 ** 32, _hash(state)
    jy = state / 2.0 ** 32
    nx, ny = (x + jx) / width * 2.0 - 1.0, (y + jy) / height * 2.0 - 1.0
    origin, target, up = (np.asarray(a, np.float64) for a in (camera.position, camera.target, camera.up))
    forward = (target - origin) / np.linalg.norm(target - origin)
    right = np.cross(forward, up)
    right /= np.linalg.norm(right)
    up = np.cross(right, forward)
    half = math.tan(math.radians(camera.vertical_fov_degrees) * 0.5)
    d = forward + nx * width / height * half * right - ny * half * up
    return origin, d / np.linalg.norm(d)


def exact(case, seed):
    """Closest hits in 64 bits for the ray queries.  A rendered frame has no
    such value: every hit and every comparison with a random number decides
    where its path goes on, so 64-bit arithmetic follows other paths."""
    if case["kind"] not in ("pick", "trace"):
        return None
    if case["kind"] == "trace":
        if float(case["width"]) * case["size"] > 3e10:
            return None
        scene, _ = _scene(case["scene"], case["size"], seed)
        corners = torch.from_numpy(scene.render_triangles()).double().cuda()
        vertices = np.concatenate([mesh.world_vertices for mesh in scene.visible_meshes])
        o, d, tmax = _rays(np.asarray(vertices, np.float32), case["width"], seed)
        hits = _closest(torch.from_numpy(o).double().cuda(), torch.from_numpy(d).double().cuda(), corners, 0.001, tmax)
        # A ray at a shared vertex or edge meets several triangles at one
        # distance: which of them is reported is no 64-bit value.
        return {"t": hits[:, 0], "u": None, "v": None, "triangle": None}
    scene, camera = _scene(case["scene"], case["size"], seed)
    w, h = case["width"], case["height"]
    px, py = _pick_pixel(case, seed)
    o, d = _pixel_ray(camera, w, h, int(px), int(py))
    corners = torch.from_numpy(scene.render_triangles()).double().cuda()
    t, u, v, triangle = _closest(torch.from_numpy(o[None]).cuda(), torch.from_numpy(d[None]).cuda(), corners, 0.001,
                                 1e30)[0]
    if triangle < 0:
        return {"object": 0, "triangle": -1, "distance": 0.0, "position": np.zeros(3), "weights": np.zeros(3)}
    return {"object": None, "triangle": None, "distance": float(t), "position": o + t * d,
            "weights": np.array([1.0 - u - v, u, v])}
