"""The frames a program renders with this library, for timing and comparing builds.

A case is one way of using the library on one scene: which scene, how large,
and which public calls take it from descriptors to results.  Scenes are those
of tetra3d_amd.workloads (the icosphere, a field of cubes, a heightfield, sets
of models of uneven size, a crowd of animated characters), at their own sizes
and at others.  Meshes and clips are assets: a program loads them once, so they
depend on the case alone.  Everything that changes between frames (placement,
armatures, playheads, lights, camera) is drawn from the seed.

Which models a camera sees depends on the case alone (the others stand behind
it), so a frame's lists have one size for every seed.  They have gaps behind
each render pair's drawn triangles that a render never writes; prepare()
clears them once, so a whole list can be compared.  Lists that go to the host
land in buffers that the program keeps.
"""
import copy
import ctypes as C
import functools
import math

import numpy as np
import torch

from tetra3d_amd import _abi as A
from tetra3d_amd import workloads as W
from tetra3d_amd.runtime import Context
from tetra3d_amd.scene import (Camera, DirectionalLight, LightVolume, Material, MeshPart, Model, PointLight, Scene,
                               Texture, World, quat_to_matrix, rotation_from_forward)
from tetra3d_amd.serving import Server

f32, f64 = np.float32, np.float64


def listed():
    return [
        # one small object in a small window: launches and the host's part of a frame are all there is
        {"name": "icosphere_642", "scene": "sphere", "level": 3, "call": "render", "width": 640, "height": 360},
        # the same kind of object rendered by a loop that may not allocate, into tensors of its own
        {"name": "icosphere_2562_noalloc", "scene": "sphere", "level": 4, "call": "noalloc", "width": 1280, "height": 720},
        # thousands of small props (crates, foliage, tiles)
        {"name": "cubes_4096", "scene": "cubes", "count": 4096, "call": "render", "width": 1920, "height": 1080},
        # one large mesh under many lights and a light volume: an outdoor level
        {"name": "terrain_1024", "scene": "terrain", "n": 1024, "call": "render", "width": 1920, "height": 1080},
        # a level of ordinary size whose lists go to a host renderer (ebiten's DrawTriangles); odd grid
        {"name": "terrain_357_host", "scene": "terrain", "n": 357, "call": "download", "width": 1280, "height": 720},
        # a full scene: models of uneven size, a quarter of them skinned; waits for each frame
        {"name": "mixed_512", "scene": "mixed", "count": 512, "vmax": 65536, "call": "render", "width": 1920, "height": 1080},
        # the same scene seen by two cameras (split screen, stereo), both frames in flight together: throughput
        {"name": "mixed_512_two_cameras", "scene": "mixed", "count": 512, "vmax": 65536, "call": "pair", "width": 1920,
         "height": 1080},
        # textures with perspective correction, transparent parts, both culling modes, a normal list
        {"name": "mixed_67_materials", "scene": "mixed", "count": 67, "vmax": 30000, "call": "render", "width": 1600,
         "height": 900, "materials": True},
        # animated characters sharing a mesh, posed on the device
        {"name": "crowd_256", "scene": "crowd", "count": 256, "bones": 64, "call": "render", "width": 1920, "height": 1080},
        # pictures instead of lists: rendered and drawn into the camera's textures
        {"name": "sphere_picture_640", "scene": "sphere", "level": 3, "call": "raster", "width": 640, "height": 360},
        {"name": "mixed_96_picture_1080", "scene": "mixed", "count": 96, "vmax": 65536, "call": "raster", "width": 1920,
         "height": 1080, "materials": True},
        # a burst of requests to a render server, each client taking its lists home
        {"name": "serve_24_jobs", "scene": "mixed", "count": 96, "vmax": 4096, "call": "serve", "jobs": 24, "width": 1280,
         "height": 720},
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    width = spread(320, 1920)
    c = {"width": width, "height": width * 9 // 16}
    scene = rng.choice(["sphere", "cubes", "terrain", "mixed", "mixed", "crowd"])
    call = rng.choice(["render", "render", "pair", "download", "raster"])
    c.update(scene=scene, call=call)
    if scene == "sphere":
        c.update(level=rng.randint(1, 6), call=rng.choice(["render", "noalloc", "pair", "download", "raster"]))
    elif scene == "cubes":
        c.update(count=spread(48, 6000))
    elif scene == "terrain":
        c.update(n=spread(24, 1000))
    elif scene == "mixed":
        c.update(count=spread(5, 300), vmax=spread(200, 50000), materials=rng.random() < 0.5)
        if rng.random() < 0.2:
            c.update(call="serve", jobs=rng.randint(3, 24), vmax=min(c["vmax"], 4000), materials=False)
    else:
        c.update(count=spread(3, 256), bones=spread(8, 100))
    if c["call"] == "download":      # lists of tens of megabytes, as a host renderer takes them
        c = {**c, **{k: min(c[k], m) for k, m in (("level", 5), ("count", 60), ("n", 500), ("vmax", 8000)) if k in c}}
    return c


# ---------------------------------------------------------------------------
# scenes
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=4)
def _asset_models(scene, level, count, n, vmax, bones):
    """The workload's models as the asset library holds them: meshes, skins, clips."""
    if scene == "sphere":
        return W.icosphere_scene(level=level).models
    if scene == "cubes":
        return [W.cube_mesh()] * count
    if scene == "terrain":
        return W.heightfield_scene(n=n).models
    if scene == "mixed":
        return W.mixed_models(W.SplitMix64(), count, vmax=vmax)
    return W.crowd_scene(count=count, bones=bones).models


def _assets(case):
    return _asset_models(case["scene"], *(case.get(k) for k in ("level", "count", "n", "vmax", "bones")))


def _rotations(rng, n):
    return [quat_to_matrix(*q) for q in W.uniform_quaternions(rng, n)]


def _places(rng, n, behind, near, far, half, fov, width, height):
    """n positions in view of a camera near the origin that looks along -z, at most `half` off its axis; the first
    `behind` of every 16 lie behind it instead."""
    depth = rng.uniform(near, far, n).astype(f64)
    slope = math.tan(math.radians(fov) / 2)
    side = rng.uniform(-1, 1, 2 * n).astype(f64).reshape(n, 2)
    x = side[:, 0] * np.minimum(half, depth * slope * width / height - 4)
    y = side[:, 1] * np.minimum(half, depth * slope)
    z = np.where(np.arange(n) % 16 < behind, depth, -depth)
    return np.stack([x, y, z], axis=1).astype(f32)


def _lights(rng, directional, points, lo, hi, ranges):
    lights = []
    for d in W.unit_vectors(rng, directional):
        sun = DirectionalLight("sun", 1, 1, 1, 1)
        sun.set_local_rotation(rotation_from_forward(d))
        lights.append(sun)
    at = np.stack([rng.uniform(lo[a], hi[a], points) for a in range(3)], axis=1) if points else []
    reach = rng.uniform(*ranges, points) if points else []
    for p, r in zip(at, reach):
        light = PointLight("point", *[float(x) for x in rng.uniform(0.4, 1, 3)], 1)
        light.set_local_position(*p)
        light.range = f32(r)
        lights.append(light)
    return lights


def _materials(models, rng):
    """Textured materials, one per model: some transparent, some cut out by their texture's alpha, some two-sided."""
    texels = (rng.floats(64 * 64 * 4) * 255).astype(np.uint8).reshape(64, 64, 4)
    texels[..., 3] = 255
    holes = texels.copy()
    holes[8:24, 8:24] = 0
    whole, cut = Texture(texels), Texture(holes)
    for m, (t, b, o) in zip(models, rng.floats(3 * len(models)).reshape(-1, 3)):
        mat = Material(m.name)
        mat.texture, mat.texture_size = whole, (64, 64)
        mat.texture_filter = A.FILTER_LINEAR if o < 0.5 else A.FILTER_NEAREST
        mat.backface_culling = bool(b < 0.8)
        if t < 0.2:
            mat.color = np.array([1, 1, 1, 0.6], dtype=f32)
        elif t < 0.3:
            mat.texture, mat.transparency_mode = cut, A.TRANSPARENCY_ALPHA_CLIP
        m.mesh = copy.copy(m.mesh)
        m.mesh.mesh_parts = [MeshPart(m.mesh, mat, 0, m.mesh.triangle_count)]


def _frames(case, seed):
    """What the seed decides: [(camera, lights, models)] of the case's Camera.Render calls, and their scene."""
    rng = W.SplitMix64(seed * 7919 + 17)
    assets = _assets(case)
    world = World()
    world.ambient_light.energy = f32(0.2)

    def camera(fov, far):
        c = Camera("camera", case["width"], case["height"])
        c.fov, c.far = f32(fov), f32(far)
        return c

    cams, models = [], []
    if case["scene"] == "sphere":
        m = copy.copy(assets[0])
        m.set_local_rotation(_rotations(rng, 1)[0])
        models = [m]
        for k in range(2):
            cam = camera(75, 100)
            cam.set_local_position(0.1 * k, 0, 4)
            cams.append(cam)
        lights = _lights(rng, 1, 1, (-2, -2, 1), (2, 2, 3), (8, 12))
    elif case["scene"] == "cubes":
        n = len(assets)
        pos = _places(rng, n, 7, 8, 200, 100, 60, case["width"], case["height"])
        scale = rng.uniform(0.5, 2, n)
        for i, r in enumerate(_rotations(rng, n)):
            m = Model("cube", assets[i])
            m.set_local_position(*pos[i])
            m.set_local_rotation(r)
            m.set_local_scale(scale[i], scale[i], scale[i])
            models.append(m)
        for k in range(2):
            cam = camera(60, 400)
            cam.set_local_position(2 * k, 0, 0)
            cams.append(cam)
        lights = _lights(rng, 1, 8, (-100, -100, -200), (100, 100, 0), (29, 31))
    elif case["scene"] == "terrain":
        m = copy.copy(assets[0])
        models = [m]
        n = case["n"]
        yaw = float(rng.floats(1)[0]) * 2 * math.pi
        for k in range(2):
            cam = camera(75, 1000)
            cam.set_local_position((n - 1) / 2 + k, 5, (n - 1) / 2)
            cam.set_local_rotation(W.axis_angle_matrix((0, 1, 0), yaw))
            cams.append(cam)
        lights = _lights(rng, 1, 16, (0, 0, 0), (n - 1, 25, n - 1), (15, 60))
        cell = min(32, (n - 1) / 4)
        volume = LightVolume("volume", *m.mesh.dimensions, (cell, 4, cell))
        volume.cells[:, :3] = rng.floats(len(volume.cells) * 3).reshape(-1, 3)
        lights.append(volume)
    elif case["scene"] == "mixed":
        n = len(assets)
        pos = _places(rng, n, 2 if n >= 32 else 0, 30, 250, 60, 50, case["width"], case["height"])
        for i, r in enumerate(_rotations(rng, n)):
            m = copy.copy(assets[i])
            m.set_local_position(*pos[i])
            m.set_local_rotation(r)
            if m.skinned:
                place = m.transform()
                angles = rng.floats(32).astype(f64) * math.radians(30)
                m.bone_influences = np.stack([W.mat_mult(W.axis_angle_matrix(a, t), place)
                                              for a, t in zip(W.unit_vectors(rng, 32), angles)]).astype(f32)
            models.append(m)
        if case.get("materials"):
            _materials(models, rng)
        for k in range(2):
            cam = camera(60, 400)
            cam.set_local_position(3 * k, 0, 0)
            if case.get("materials"):
                cam.perspective_corrected_texture_mapping = True
                cam.render_normals = case["call"] != "raster"
            cams.append(cam)
        lights = _lights(rng, 1, 8, (-60, -60, -250), (60, 60, -30), (79, 81))
    else:
        n = len(assets)
        clips = {}
        heads = rng.uniform(-0.1, 1.1, n)
        for i, r in enumerate(_rotations(rng, n)):
            m = copy.copy(assets[i])
            m.set_local_position(-30 + 4 * (i % 16), -6 + 4 * ((i // 16) % 4), -40 - 6 * (i // 64))
            m.set_local_rotation(r)
            m.armature_parent = m.transform()
            clip = m.animation
            if id(clip) not in clips:
                clips[id(clip)] = copy.copy(clip)
                clips[id(clip)].handle = 0        # a copy of its own for this program's context
            m.animation = clips[id(clip)]
            m.animation_time = float(heads[i])
            models.append(m)
        for k in range(2):
            cam = camera(60, 400)
            cam.set_local_position(k, 0, 0)
            cams.append(cam)
        lights = _lights(rng, 1, 4, (-30, -8, -60), (30, 8, -30), (59, 61))
    scene = Scene(case["scene"], world)
    if case["call"] == "serve":
        jobs, asked = [], W.SplitMix64(case["jobs"])      # what each client asks for is the case's
        for j in range(case["jobs"]):
            ids = np.unique(asked.ints(0, len(models), int(asked.ints(1, 13, 1)[0])))
            few = lights[: 1 + int(asked.ints(0, len(lights), 1)[0])]
            jobs.append((camera(50 + 30 * float(rng.floats(1)[0]), 400), few, [models[i] for i in ids]))
        return jobs, scene
    return [(cam, lights, models) for cam in cams[: 2 if case["call"] == "pair" else 1]], scene


# ---------------------------------------------------------------------------
# one program's state and one pass
# ---------------------------------------------------------------------------

class _Span:
    """Device memory of a frame as torch sees it; holds the context that owns it."""

    def __init__(self, address, shape, kind, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": kind, "data": (address, False), "version": 2}


def _tensor(address, shape, kind, owner):
    return torch.as_tensor(_Span(address, shape, kind, owner), device="cuda")


class _Lists:
    """A frame's device lists: tensors over the arrays that t3d_frame_device_outputs names."""

    def __init__(self, ctx, frame, normals):
        self.ctx, self.frame, self.normals = ctx, frame, normals
        self.at, self.out = None, {}
        self.ptr = [C.c_void_p() for _ in range(4)]

    def __call__(self):
        L = self.ctx.L
        self.ctx._check(L.t3d_frame_device_outputs(self.frame, *[C.byref(p) for p in self.ptr[:3]]))
        if self.normals:
            self.ctx._check(L.t3d_frame_device_normals(self.frame, C.byref(self.ptr[3])))
        pairs = _pairs(self.ctx, self.frame)
        at = tuple(p.value for p in self.ptr)
        if at != self.at:
            room = max((int(p[4]) + (int(p[5]) << 32) + 3 * int(p[2]) for p in pairs), default=0)
            kinds = {"color": "<f4", "depth": "<f4", "indices": "<i4", "normals": "<f4"}   # corner numbers are below 2^31
            self.out = {name: _tensor(address, (room, 12) if kind == "<f4" else (room,), kind, self.ctx)
                        for (name, kind), address in zip(kinds.items(), at) if address and room}
            self.at = at
        return {"pairs": pairs, **self.out}


def _pairs(ctx, frame):
    """t3d_frame_pairs: model, part, triangles, drawn triangles and first vertex (two words) of every render pair."""
    n = C.c_uint32()
    ptr = C.POINTER(A.PairResult)()
    ctx._check(ctx.L.t3d_frame_pairs(frame, C.byref(n), C.byref(ptr)))
    if not n.value:
        return np.zeros((0, 6), dtype=np.int64)
    raw = (C.c_uint8 * (n.value * C.sizeof(A.PairResult))).from_address(C.addressof(ptr.contents))
    return np.frombuffer(raw, dtype=np.uint32).reshape(n.value, 6).astype(np.int64)


def prepare(case, seed):
    frames, scene = _frames(case, seed)
    ctx = Context(0)
    everything = [m for _, _, models in frames for m in models]
    lights = [l for _, ls, _ in frames for l in ls]
    ctx.prepare(_Everything(everything, lights))
    inputs = [ctx.inputs(cam, scene, ls, models) for cam, ls, models in frames]
    state = {"call": case["call"], "ctx": ctx, "inputs": inputs, "frames": [ctx.frame]}
    if case["call"] == "pair":
        state["frames"].append(ctx.new_frame())
    tris = sum(m.mesh.triangle_count for m in everything)
    if case["call"] == "noalloc":
        state["own"] = {"color": torch.zeros((3 * tris, 12), device="cuda"),
                        "depth": torch.zeros((3 * tris, 12), device="cuda"),
                        "indices": torch.zeros(3 * tris, dtype=torch.int32, device="cuda")}
        torch.cuda.synchronize()
    elif case["call"] in ("download", "serve"):
        own = {"color": torch.zeros((3 * tris, 12), pin_memory=True), "depth": torch.zeros((3 * tris, 12), pin_memory=True),
               "indices": torch.zeros(3 * tris, dtype=torch.int32, pin_memory=True)}
        if case["call"] == "serve":
            own["triangles"] = torch.zeros(tris, dtype=torch.int32, pin_memory=True)
            state["server"] = _Server(ctx, slots=4, max_batch_jobs=16, hbm_budget=0)
            state["job_pairs"] = (A.PairResult * max(len(models) for _, _, models in frames))()
        elif frames[0][0].render_normals:
            own["normals"] = torch.zeros((3 * tris, 12), pin_memory=True)
        state["own"] = own
    if case["call"] in ("render", "pair"):
        normals = bool(frames[0][0].render_normals)
        state["lists"] = [_Lists(ctx, f, normals) for f in state["frames"]]
        for frame, inp, lists in zip(state["frames"], inputs, state["lists"]):
            ctx.render_async(inp, frame)
            ctx.wait(frame)
            for name, t in lists().items():
                if name != "pairs":
                    t.zero_()
        torch.cuda.synchronize()
    return state


class _Server(Server):
    """A server that ends with the state that holds it, before its context."""

    def __del__(self):
        self.close()


class _Everything:
    """The assets of several Camera.Render calls, as Context.prepare takes a workload's."""

    def __init__(self, models, lights):
        def once(values):
            return list({id(v): v for v in values if v is not None}.values())
        self.models = models
        self.meshes = once(m.mesh for m in models)
        self.volumes = once(l for l in lights if isinstance(l, LightVolume))
        self.animations = once(m.animation for m in models)


def run(state):
    ctx, inputs, call = state["ctx"], state["inputs"], state["call"]
    if call == "render":
        ctx.render_inputs(inputs[0])
        return state["lists"][0]()
    if call == "pair":
        for frame, inp in zip(state["frames"], inputs):
            ctx.render_async(inp, frame)
        out = []
        for frame, lists in zip(state["frames"], state["lists"]):
            ctx.wait(frame)
            out.append(lists())
        return out
    own = state.get("own")
    if call == "noalloc":
        ctx.render_noalloc(inputs[0], own["color"].data_ptr(), own["depth"].data_ptr(), own["indices"].data_ptr(),
                           len(own["indices"]))
        return {"pairs": _pairs(ctx, ctx.frame), **own}
    if call == "download":
        ctx.render_inputs(inputs[0])
        ctx._check(ctx.L.t3d_frame_download(ctx.ctx, ctx.frame, _vertices(own["color"]), _vertices(own["depth"]),
                                            _words(own["indices"])))
        if "normals" in own:
            ctx._check(ctx.L.t3d_frame_download_normals(ctx.ctx, ctx.frame, _vertices(own["normals"])))
        return {"pairs": _pairs(ctx, ctx.frame), **own}
    if call == "raster":
        ctx.render_inputs(inputs[0])
        ctx.rasterize()
        color, depth = ctx.download_images()
        return {"color": color, "depth": depth}
    server, at = state["server"], 0
    jobs = [server.submit_inputs(inp) for inp in inputs]
    server.drain()
    for job in jobs:
        server._check(server.L.t3d_job_download(server.srv, job, state["job_pairs"], _vertices(own["color"], 3 * at),
                                                _vertices(own["depth"], 3 * at), _words(own["indices"], 3 * at),
                                                _words(own["triangles"], at)))
        at += int(server.info(job).survivors)
    for job in jobs:
        server.release(job)
    return own


def _vertices(t, first=0):
    return C.cast(t.data_ptr() + 48 * first, C.POINTER(A.Vertex))


def _words(t, first=0):
    return C.cast(t.data_ptr() + 4 * first, C.POINTER(C.c_uint32))


# What share of a scene's triangles a frame draws, about: culling by the frustum and of back faces.
_DRAWN = {"sphere": 0.37, "cubes": 0.26, "terrain": 0.135, "mixed": 0.44, "crowd": 0.4}


def work(case):
    """Mesh streams read once (position, normal, colour, UV, skin, indices), palettes, and each output written once."""
    assets = _assets(case)
    points = {"sphere": 2, "cubes": 9, "terrain": 18, "mixed": 9, "crowd": 5}[case["scene"]]
    read = verts = tris = 0
    for a in assets:
        mesh = getattr(a, "mesh", a)
        v, t = mesh.vertex_count, mesh.triangle_count
        per = 32 + (16 if mesh.colors is not None else 0) + (24 if mesh.bone_indices is not None else 0)
        verts, tris = verts + v, tris + t
        read += v * per + t * (6 if v <= 65536 else 12)
    read += 64 * case.get("bones", 0) * len(assets)
    calls = {"pair": 2, "serve": case.get("jobs", 0) * 6.5 / len(assets)}.get(case["call"], 1)
    drawn = _DRAWN[case["scene"]] * tris
    bytes_ = read + drawn * (300 + (144 if case.get("materials") and case["call"] == "render" else 0))
    flops = verts * (60 + 40 * points) + tris * 30 + drawn * 60
    if case["call"] == "raster":
        pixels = case["width"] * case["height"]
        bytes_, flops = read + 8 * pixels, flops + 400 * pixels
    return {"bytes": calls * bytes_, "flops": calls * flops}


# ---------------------------------------------------------------------------
# the same lists in 64 bits
# ---------------------------------------------------------------------------
# What a frame draws and in which order are decisions on float32 numbers (a
# cull test, one of 512 depth bins, a light volume's cell), and 64 bits would
# decide some of them otherwise.  They are taken here in float32, operation by
# operation; every number in a list is then computed in float64 throughout.

def _mult(a, b):
    return ((a[:, 0:1] * b[0:1] + a[:, 1:2] * b[1:2]) + a[:, 2:3] * b[2:3]) + a[:, 3:4] * b[3:4]


def _inverse(m):
    """By cofactors, in the order that a float32 program would take."""
    def minor(r, c):
        return m[r[0], c[0]] * m[r[1], c[1]] - m[r[0], c[1]] * m[r[1], c[0]]

    def cofactor(i, j):
        r, c = [k for k in range(4) if k != i], [k for k in range(4) if k != j]
        return (m[r[0], c[0]] * minor(r[1:], c[1:]) - m[r[0], c[1]] * minor(r[1:], (c[0], c[2]))
                + m[r[0], c[2]] * minor(r[1:], c[:2]))

    det = m.dtype.type(1) / (m[0, 0] * cofactor(0, 0) - m[0, 1] * cofactor(0, 1) + m[0, 2] * cofactor(0, 2)
                             - m[0, 3] * cofactor(0, 3))
    out = np.empty((4, 4), dtype=m.dtype)
    for i in range(4):
        for j in range(4):
            c = cofactor(j, i)
            out[i, j] = det * (-c if (i + j) % 2 else c)
    return out


def _length(v):
    return np.sqrt(v[..., 0] * v[..., 0] + v[..., 1] * v[..., 1] + v[..., 2] * v[..., 2])


def _unit(v):
    length = _length(v)[..., None]
    with np.errstate(all="ignore"):
        return np.where((length < 1e-8) | (length == 1), v, v / length)


def _decompose(m):
    rot = np.eye(4, dtype=m.dtype)
    rot[:3, :3], rot[:3, 3] = _unit(m[:3, :3]), m[:3, 3]
    return m[3, :3], _length(_mult(m, np.ascontiguousarray(rot.T))[:3, :3]), rot


def _into(model, world):
    """A world position in a model's space: its inverse's rotation, and its translation over its scale."""
    p, s, r = _decompose(_inverse(model))
    return _point(r, world) + p * (world.dtype.type(1) / s)


def _point(m, v, w=False):
    """v @ m with m's translation, columns x, y, z (and w)."""
    return np.stack([((m[0, j] * v[..., 0] + m[1, j] * v[..., 1]) + m[2, j] * v[..., 2]) + m[3, j]
                     for j in range(4 if w else 3)], axis=-1)


def _dot(a, b):
    return a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1] + a[..., 2] * b[..., 2]


def _view_projection(cam, kind):
    near, far, fov = kind(cam.near), kind(cam.far), kind(cam.fov)
    t = kind(math.tan(float(fov * kind(math.pi) / kind(360))))
    r = t * (kind(cam.width) / kind(cam.height))
    p = np.zeros((4, 4), dtype=kind)
    p[0, 0], p[1, 1], p[3, 2] = kind(2) * near / (r + r), kind(2) * near / (t + t), -1
    p[2, 2], p[2, 3] = -((far + near) / (far - near)), -(kind(2) * far * near / (far - near))
    turn, at = cam.world_rotation().astype(kind), cam.transform()[3, :3].astype(kind)
    move = np.eye(4, dtype=kind)
    move[3, :3] = -at
    view = _mult(move, np.ascontiguousarray(turn.T))
    return view, _mult(view, p)


def _in_frustum(cam, model):
    position, scale, rot = _decompose(model.transform().astype(f64))
    lo, hi = (d.astype(f64) for d in model.mesh.dimensions)
    centre = np.zeros(3) if model.skinned else (lo + hi) / 2
    diff = position + _point(rot, centre) * scale - cam.transform()[3, :3]
    radius = _length((hi - lo) * scale) / 2
    right, up, forward = (_unit(cam.world_rotation()[k, :3].astype(f64)) for k in range(3))
    z = -_dot(diff, forward)
    if z > cam.far + radius or z < cam.near - radius:
        return False
    angle, aspect = cam.fov * f32(3.1415) / 360, cam.width / cam.height
    tan = math.tan(angle)
    z *= tan
    if abs(_dot(diff, up)) > z + radius / math.cos(angle):
        return False
    return abs(_dot(diff, right)) <= z * aspect + radius / math.cos(math.atan(tan * aspect))


def _skin(mesh, palette, kind):
    """Positions and normals under the weighted bones."""
    palette, pos, nrm = palette.astype(kind), mesh.positions.astype(kind), mesh.normals.astype(kind)
    m = np.zeros((len(pos), 4, 4), dtype=kind)
    for k in range(4):
        m += palette[mesh.bone_indices[:, k]] * mesh.bone_weights[:, k].astype(kind)[:, None, None]
    def through(v, row3):
        return np.stack([((m[:, 0, j] * v[:, 0] + m[:, 1, j] * v[:, 1]) + m[:, 2, j] * v[:, 2]) + row3(j)
                         for j in range(3)], axis=-1)
    return through(pos, lambda j: m[:, 3, j]), through(nrm, lambda j: kind(0))


def _volume_cells(light, world):
    """A light volume's colour at float32 world positions, black outside it."""
    lo, size = light.dims_min, light.cell_size
    inside = np.all((world >= lo) & (world <= light.dims_max), axis=1)
    q = (((world - light.offset) - lo) - size / f32(2)) / size
    cell = (np.sign(q) * np.floor(np.abs(q).astype(f64) + 0.5)).astype(np.int64)
    count = np.array(light.cell_count)
    inside &= np.all((cell >= 0) & (cell < count), axis=1)
    cell[~inside] = 0
    at = cell[:, 0] + cell[:, 1] * count[0] + cell[:, 2] * count[0] * count[1]
    return np.where(inside[:, None], light.cells[at, :3].astype(f64) if len(light.cells) else 0.0, 0.0)


def _lit(model, lights, ambient, pos, nrm, pos32):
    """The light that reaches each vertex, in the space its positions are given in."""
    total = np.zeros((len(pos), 3)) + ambient
    base = model.transform().astype(f64)
    for light in lights:
        color = light.color.astype(f64)
        if light.TYPE == A.LIGHT_POINT:
            at, reach = light.transform()[3, :3].astype(f64), float(light.range)
            to = (at if model.skinned else _into(base, at)) - pos
            d2 = _dot(to, to)
            far = d2 > reach * reach
            diffuse = np.maximum(_dot(nrm, _unit(to)), 0)
            with np.errstate(divide="ignore"):
                f = diffuse * (2 / (1 + 0.1 * d2)) * np.clip((reach * reach - d2) / d2, 0, 1)
            total += np.where(far, 0, f)[:, None] * color * float(light.energy)
        elif light.TYPE == A.LIGHT_DIRECTIONAL:
            way = light.world_rotation()[2, :3].astype(f64)
            turned = nrm if model.skinned else _point(
                np.ascontiguousarray(_inverse(model.world_rotation().astype(f64)).T), nrm)
            total += np.maximum(_dot(turned, _unit(way)), 0)[:, None] * color * float(light.energy)
        else:
            world = pos32 if model.skinned else _point(model.transform(), pos32)
            total += _volume_cells(light, world) * color * float(light.energy)
    return total


def _draw_pair(cam, scene, lights, model, normals):
    """One model's colour, depth (and normal) lists and its drawn triangles, farthest bin first."""
    mesh, mat = model.mesh, model.mesh.mesh_parts[0].material
    tri = mesh.indices.astype(np.int64)
    (_, vp32), (view, vp) = _view_projection(cam, f32), _view_projection(cam, f64)
    base32, base = model.transform(), model.transform().astype(f64)
    eye32 = cam.transform()[3, :3]
    if model.skinned:
        pos32, (pos, nrm) = _skin(mesh, model.bone_influences, f32)[0], _skin(mesh, model.bone_influences, f64)
        clip32, clip = _point(vp32, pos32, True), _point(vp, pos, True)
    else:
        pos32, pos, nrm = mesh.positions, mesh.positions.astype(f64), mesh.normals.astype(f64)
        clip32, clip = _point(_mult(base32, vp32), pos32, True), _point(_mult(base, vp), pos, True)
    # which triangles, in which order (float32)
    with np.errstate(all="ignore"):
        w = np.where(clip32[:, 3] < 0, f32(0.000001), clip32[:, 3])
        x, y = (clip32[:, 0] / w)[tri], (clip32[:, 1] / w)[tri]
        keep = ((clip32[:, 2] + f32(1) >= cam.near) & (clip32[:, 2] < cam.far))[tri].any(axis=1)
        for v in (x, y):
            keep &= ~((v < -0.5).all(axis=1) | (v > 0.5).all(axis=1))
        if mat.backface_culling:
            keep &= ~((x[:, 0] - x[:, 1]) * (y[:, 1] - y[:, 2]) - (x[:, 1] - x[:, 2]) * (y[:, 0] - y[:, 1]) < 0)
        corners = pos32[tri]
        centre = ((corners[:, 0] + corners[:, 1]) + corners[:, 2]) / f32(3)
        d = (eye32 if model.skinned else _into(base32, eye32)) - centre
        key = _dot(d, d)
        keep &= np.isfinite(key)
    ids = np.flatnonzero(keep)
    key = key[ids]
    if len(ids):
        low, span = key.min(), key.max() - key.min()
        span = span + f32(0.001) if span == 0 else span
        bins = np.clip((key - low) / span * f32(512), 0, 511).astype(np.int64)
        ids = ids[np.argsort(511 - bins, kind="stable")]
    # their numbers (float64)
    world = scene.world
    tint = model.color.astype(f64) * mat.color.astype(f64)
    paint = np.ones((len(pos), 4)) * tint
    if mesh.colors is not None:
        paint = mesh.colors.astype(f64) * tint
    light = _lit(model, lights, float(world.ambient_light.energy), pos, nrm, pos32)
    paint[:, :3] *= light
    w = np.where(clip[:, 3] < 0, 0.001, clip[:, 3])
    out = np.zeros((len(pos), 12))
    with np.errstate(divide="ignore"):       # a vertex may lie on the eye's plane
        out[:, 0] = clip[:, 0] / w * cam.width + cam.width / 2
        out[:, 1] = clip[:, 1] / -w * cam.height + cam.height / 2
    size = mat.texture_size or (0, 0)
    uv = mesh.uvs.astype(f64)
    over = w if cam.perspective_corrected_texture_mapping else 1.0
    out[:, 2], out[:, 3] = uv[:, 0] / over * size[0], (1 - uv[:, 1]) / over * size[1]
    if cam.perspective_corrected_texture_mapping:
        out[:, 8] = 1 / w
    lists = {"color": out, "depth": out.copy()}
    out[:, 4:8] = paint
    margin = float(cam.far - cam.near) * float(cam.depth_margin)
    deep = np.clip((clip[:, 2] + margin) / (float(cam.far - cam.near) + margin * 2), 0, 1)
    lists["depth"][:, 4:7], lists["depth"][:, 7] = deep[:, None], 1
    if normals:
        turned = _point(_decompose(_mult(base, view))[2], pos)
        lists["normals"] = np.concatenate([out[:, :4], turned * 0.5 + 0.5, np.zeros((len(pos), 5))], axis=1)
    drawn = tri[ids].ravel()
    return {name: values[drawn] for name, values in lists.items()}


def _pairs_in_order(cam, models):
    """The models in the frustum: opaque ones as listed, then transparent ones, farthest first."""
    seen = [m for m in models if _in_frustum(cam, m)]

    def clear(m):
        mat = m.mesh.mesh_parts[0].material
        return mat.transparency_mode == A.TRANSPARENCY_AUTO and mat.color[3] < 0.999

    def distance(m):
        d = cam.transform()[3, :3] - m.transform()[3, :3]
        return -_dot(d, d)
    return [m for m in seen if not clear(m)] + sorted((m for m in seen if clear(m)), key=distance)


def exact(case, seed):
    if case["scene"] == "crowd" or case["call"] == "raster":
        return None             # animated armatures; pictures of whole bytes
    if sum(getattr(a, "mesh", a).triangle_count for a in _assets(case)) > 2_500_000:
        return None             # over 20 seconds
    frames, scene = _frames(case, seed)
    gaps = case["call"] not in ("download", "serve")
    out = []
    for cam, lights, models in frames:
        names = ["color", "depth"] + (["normals"] if cam.render_normals else [])
        lists = {name: [] for name in names}
        order = _pairs_in_order(cam, models)
        for m in order:
            drawn = _draw_pair(cam, scene, lights, m, cam.render_normals)
            for name in names:
                lists[name].append(drawn[name])
                if gaps:
                    lists[name].append(np.zeros((3 * m.mesh.triangle_count - len(drawn[name]), 12)))
        out.append({name: np.concatenate(v or [np.zeros((0, 12))]) for name, v in lists.items()})
    if case["call"] == "pair":
        return out
    if gaps and case["call"] != "noalloc":
        return out[0]
    tris = sum(m.mesh.triangle_count for _, _, models in frames for m in models)   # the caller's own arrays
    lists = {name: np.zeros((3 * tris, 12)) for name in out[0]}
    for name, values in lists.items():
        whole = np.concatenate([f[name] for f in out])
        values[: len(whole)] = whole
    return lists
