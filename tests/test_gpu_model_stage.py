"""The model-level stage of Camera.Render on the device (k_models and
k_plist: the frustum spheres of model.go:142-182 against SphereInFrustum,
camera.go:933-983; the render pairs of camera.go:1343-1457 with the
transparents' stable sort of camera.go:2050-2055) bit for bit against the
oracle, and against the host build of the same frames."""
import numpy as np
import pytest

from tetra3d_amd import _abi as A
from tetra3d_amd import workloads as W
from tetra3d_amd.runtime import Context
from tetra3d_amd.scene import Material, Model, Scene, World, DirectionalLight, Camera
from tests.feature_scenes import feature_scene, pair_order_scene
from tests.parity import compare_frames

f32 = np.float32


def _with_stage(gpu_ctx, on):
    saved = gpu_ctx.tuning()
    gpu_ctx.set_tuning(model_stage=int(on))
    return saved


@pytest.mark.gpu
def test_stage_runs_where_it_applies(gpu_ctx, oracle):
    """With the stage on, a frame with RenderDepth and no dynamic batch runs
    k_models; with it off, or with RenderDepth off, the host builds the pairs."""
    wl = pair_order_scene(1)      # odd seeds render depth
    wl_nodepth = pair_order_scene(0)
    saved = gpu_ctx.tuning()
    try:
        for on, scene, expect in ((1, wl, True), (0, wl, False), (1, wl_nodepth, False)):
            gpu_ctx.set_tuning(model_stage=on)
            gpu_ctx.profile(True)
            gpu_ctx.profile_read(reset=True)
            g = gpu_ctx.render_workload(scene)
            prof = gpu_ctx.profile_read(reset=True)
            gpu_ctx.profile(False)
            print("stage", on, scene.name, sorted(prof), flush=True)
            assert ("k_models" in prof) == expect
            compare_frames(g, oracle.render_workload(scene))
    finally:
        gpu_ctx.profile(False)
        gpu_ctx.L.t3d_set_tuning(gpu_ctx.ctx, saved)


@pytest.mark.gpu
def test_tuning_round_trip():
    """A small frame is built on the host as a context starts; setting the tuning that the context has, or another field
    of it, changes nothing about that; model_stage 1 takes the frame to the device, and what was saved takes it back."""
    wl = pair_order_scene(1)
    with Context(0) as ctx:
        def staged():
            ctx.profile(True)
            ctx.profile_read(reset=True)
            ctx.render_workload(wl)
            ctx.profile(False)
            return "k_models" in ctx.profile_read(reset=True)

        saved = ctx.tuning()
        print("tuning round trip", saved.model_stage, flush=True)
        assert not staged()
        ctx.set_tuning()
        assert not staged()
        ctx.set_tuning(store_mode=18)
        assert not staged()
        ctx.set_tuning(use_graph=1)           # a graph wants launches that stay the same: the device's
        assert staged()
        ctx.set_tuning(use_graph=0)
        assert not staged()
        ctx.set_tuning(model_stage=1)
        assert staged()
        ctx._check(ctx.L.t3d_set_tuning(ctx.ctx, saved))
        assert not staged()


@pytest.mark.gpu
@pytest.mark.parametrize("on", [0, 1], ids=["host", "device"])
def test_feature_scenes_host_build(gpu_ctx, oracle, on):
    """The feature scenes built on the host whatever their size, and by the
    stage where it applies (as a context starts, scenes so small are left to
    the host)."""
    saved = _with_stage(gpu_ctx, on)
    try:
        for seed in range(40):
            wl = feature_scene(seed)
            print("feature scene", seed, "stage", on, flush=True)
            compare_frames(gpu_ctx.render_workload(wl), oracle.render_workload(wl))
    finally:
        gpu_ctx.L.t3d_set_tuning(gpu_ctx.ctx, saved)


def _transparent_field(seed, n, spots=6):
    """n small spheres on a few shared positions (equal camera distances),
    most transparent with render orders -2..2, some opaque, some materials
    hidden, some models outside the frustum: the device's ranking of the
    transparents rests on the stable tie order."""
    rng = np.random.default_rng(seed)
    cam = Camera("cam", 640, 360)
    cam.render_depth = True
    where = rng.uniform([-6, -4, -30], [6, 4, -4], (spots, 3)).astype(f32)
    lights = [DirectionalLight("sun", 1, 1, 1, 1.0)]
    lights[0].set_local_rotation(W.axis_angle_matrix((1, 0, 0), -0.6))
    models = []
    for i in range(n):
        mesh = W.icosphere(0, 0.5, name="s%d" % i)   # materials belong to mesh parts: one mesh each
        m = Model("m%d" % i, mesh)
        mat = Material("mat%d" % i)
        transparent = rng.random() < 0.7
        mat.color = np.array([*rng.uniform(0.3, 1, 3), 0.5 if transparent else 1.0], dtype=f32)
        mat.render_order = int(rng.integers(-2, 3))
        mat.visible = bool(rng.random() > 0.05)
        for p in mesh.mesh_parts:
            p.material = mat
        if rng.random() < 0.1:
            m.set_local_position(0, 0, 50)   # behind the camera
        else:
            m.set_local_position(*where[rng.integers(0, spots)])
        models.append(m)
    world = World()
    world.ambient_light.energy = f32(0.3)
    return W.Workload("transparent_field_%d" % seed, cam, Scene("tf", world), lights, models)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [40, 1500])
def test_transparent_order_on_device(gpu_ctx, oracle, n):
    """Hundreds of transparents at shared distances with several render
    orders, in one and in more than one 1024-candidate chunk of k_plist."""
    saved = _with_stage(gpu_ctx, 1)
    try:
        for seed in range(2):
            wl = _transparent_field(seed, n)
            print("transparent field", seed, n, flush=True)
            s = compare_frames(gpu_ctx.render_workload(wl), oracle.render_workload(wl))
            assert s["pairs"] > 0
    finally:
        gpu_ctx.L.t3d_set_tuning(gpu_ctx.ctx, saved)


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [0, 1], ids=["direct", "graph"])
def test_cubes_camera_turning(gpu_ctx, oracle, graph):
    """4,096 cubes under a turning camera: the visible set changes every
    frame while the launch shape (sized for every cube drawn), and with it a
    graph of the launches, stays the same."""
    wl = W.cubes_scene()
    counts = []
    saved = gpu_ctx.tuning()
    gpu_ctx.set_tuning(use_graph=graph)
    try:
        for k, yaw in enumerate([0.0, 0.4, 1.3, 3.0]):
            wl.camera.set_local_rotation(W.axis_angle_matrix((0, 1, 0), yaw))
            print("cubes frame", k, "yaw", yaw, "graph", graph, flush=True)
            s = compare_frames(gpu_ctx.render_workload(wl), oracle.render_workload(wl))
            counts.append(s["pairs"])
    finally:
        gpu_ctx.L.t3d_set_tuning(gpu_ctx.ctx, saved)
    assert len(set(counts)) > 1
