"""Frames at and one past the model counts where the pairs stop being built on the host, the uniforms stop coming from
it and the tile tables start, on a context whose tuning nobody has set, against the oracle bit for bit; and their
lists downloaded with and without the triangle ids."""
import ctypes as C

import numpy as np
import pytest

from tetra3d_amd import workloads as W
from tetra3d_amd.runtime import Context
from tetra3d_amd.scene import Camera, Model, Scene
from tests.parity import compare_frames
from tests.test_gpu_pairs import _mesh


@pytest.fixture(scope="module")
def fresh_ctx():
    with Context(0) as c:
        c.poison_outputs(0x7FC0DEAD)
        yield c


@pytest.mark.gpu
@pytest.mark.parametrize("large", [False, True], ids=["small", "large"])
@pytest.mark.parametrize("count", [1, 4, 5, 16, 17, 192, 193, 640, 641])
def test_model_counts(fresh_ctx, oracle, count, large):
    r = np.random.default_rng(count)
    meshes = [_mesh(64, 60, 1), _mesh(300, 500, 2), _mesh(3000, 5000, 3)][: 3 if large else 2]
    models = []
    for i in range(count):
        m = Model("m%d" % i, meshes[-1 if i % 40 == 0 else i % 2])
        m.set_local_position(*(r.uniform(-4, 4, 3) - [0, 0, 6]))
        m.color = np.array([*r.random(3), 0.5 if i % 11 == 3 else 1.0], dtype=np.float32)
        m.shadeless = i % 7 == 5
        models.append(m)
    W._skin(models[count // 2], W.SplitMix64(5), bones=8)
    wl = W.Workload("few", Camera("camera", 800, 450), Scene("few", W._world(0.2)), W.icosphere_scene().lights, models)
    print("few models", count, large, flush=True)
    got, want = fresh_ctx.render_workload(wl), oracle.render_workload(wl)
    compare_frames(got, want)
    lists = fresh_ctx.download(triangles=False)
    for name in ("color", "depth"):
        np.testing.assert_array_equal(getattr(lists, name).view(np.uint32), getattr(want, name).view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("count,graph", [(799, 0), (801, 0), (801, 1)])
def test_large_frames_in_flight(fresh_ctx, oracle, count, graph):
    """Two frames of just under and just over 2.4 million vertices in flight, which overlap on the device or run in
    turn, launched directly or from a graph: each equals the oracle's."""
    mesh = _mesh(3000, 5000, 3)
    r = np.random.default_rng(count)
    models = []
    for i in range(count):
        m = Model("m%d" % i, mesh)
        m.set_local_position(*(r.uniform(-4, 4, 3) - [0, 0, 6]))
        m.frustum_culling = False          # all of them drawn: what counts is the drawn pairs' vertices
        models.append(m)
    lights = W.icosphere_scene().lights
    frames = [fresh_ctx.frame, fresh_ctx.new_frame()]
    wls = []
    for k in range(2):
        cam = Camera("camera%d" % k, 800, 450)
        cam.set_local_position(0.3 * k, 0, 0)
        wls.append(W.Workload("large", cam, Scene("large", W._world(0.2)), lights, models))
    fresh_ctx.prepare(wls[0])
    inputs = [fresh_ctx.inputs(w.camera, w.scene, w.lights, w.models) for w in wls]
    print("large frames in flight", count, graph, flush=True)
    saved = fresh_ctx.tuning()
    fresh_ctx.set_tuning(use_graph=graph)
    try:
        for _ in range(2):
            for f, inp in zip(frames, inputs):
                fresh_ctx.render_async(inp, f)
    finally:
        fresh_ctx.L.t3d_set_tuning(fresh_ctx.ctx, saved)
    for f, w in zip(frames, wls):
        fresh_ctx.wait(f)
        compare_frames(fresh_ctx.download(frame=f), oracle.render_workload(w))


@pytest.mark.gpu
@pytest.mark.parametrize("stage", [0, 1], ids=["host", "device"])
@pytest.mark.parametrize("shown,turns", [(40, 0), (799, 0), (801, 1)])
def test_what_is_drawn_decides_who_takes_turns(fresh_ctx, shown, turns, stage):
    """820 models listed, 2.46 million vertices in all: their frames take turns only when over 2.4 million are drawn, by
    the drawn pairs of a host-built frame or of a device-built one's last render; a frame that is waited for never does."""
    mesh = _mesh(3000, 5000, 3)
    models = []
    for i in range(820):
        m = Model("m%d" % i, mesh)
        m.set_local_position(0.01 * (i % 100), 0, -6 if i < shown else 300)
        models.append(m)
    wl = W.Workload("listed", Camera("camera", 800, 450), Scene("listed", W._world(0.2)), W.icosphere_scene().lights, models)
    fresh_ctx.prepare(wl)
    inp = fresh_ctx.inputs(wl.camera, wl.scene, wl.lights, wl.models)
    frame, out = fresh_ctx.new_frame(), C.c_int32()

    def in_turn():
        assert fresh_ctx.L.t3d_debug_frame_in_turn(frame, C.byref(out)) == 0
        return out.value

    print("drawn of the listed", shown, stage, flush=True)
    saved = fresh_ctx.tuning()
    fresh_ctx.set_tuning(model_stage=stage)
    try:
        for k in range(2):
            fresh_ctx.render_async(inp, frame)
            assert in_turn() == (turns if k or not stage else 0)
            fresh_ctx.wait(frame)
            assert len(fresh_ctx.pairs(frame)) == shown
        fresh_ctx._check(fresh_ctx.L.t3d_render(fresh_ctx.ctx, frame, C.byref(inp.render)))
        assert in_turn() == 0
    finally:
        fresh_ctx.L.t3d_set_tuning(fresh_ctx.ctx, saved)
