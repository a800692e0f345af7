"""What a frame takes of its context's memory budget."""
import numpy as np
import pytest

from tetra3d_amd import _abi as A
from tetra3d_amd import workloads as W
from tetra3d_amd.runtime import Context
from tetra3d_amd.scene import Camera, LightVolume, Model, Scene
from tetra3d_amd.serving import Server
from tests.parity import compare_frames
from tests.test_gpu_assembly import _strip
from tests.test_gpu_pairs import _mesh


def _prepared(ctx, wl):
    for m in wl.meshes:
        m._handles.pop("gpu", None)       # of an earlier context
    ctx.prepare(wl)


@pytest.mark.gpu
def test_few_pairs_take_no_more_than_plain(oracle):
    """A frame of few pairs, whose uniforms are in its tables, takes as much as the same frame with a chain for each
    pair, which has them in its scratch (each buffer is a multiple of 64 KiB: over several sizes, on average)."""
    extra = []
    for count in range(150, 186, 5):
        models = []
        for i in range(count):
            m = Model("m%d" % i, _mesh(3, 1, 1))
            m.frustum_culling = False
            models.append(m)
        wl = W.Workload("few", Camera("camera", 320, 180), Scene("few", W._world(0.2)),
                        W.icosphere_scene().lights * 5, models)
        used = []
        for mode in (A.EXEC_BATCHED, A.EXEC_PLAIN):
            with Context(0) as ctx:
                _prepared(ctx, wl)
                before = ctx.memory_used
                ctx.render_inputs(ctx.inputs(wl.camera, wl.scene, wl.lights, wl.models, mode))
                used.append(ctx.memory_used - before)
                compare_frames(ctx.download(), oracle.render_workload(wl))
        print("budget of few pairs", count, used, flush=True)
        extra.append(used[0] - used[1])
    assert np.mean(extra) <= 32 << 10


def _flat_shaded(counts, skinned, normals=False):
    """Models of separate triangles (three vertices each), as flat shading needs them; `skinned` of every four skinned."""
    models = []
    for i, n in enumerate(counts):
        m = Model("m%d" % i, _strip(n, "strip%d" % i))
        m.frustum_culling = False
        if i % 4 < skinned:
            W._skin(m, W.SplitMix64(5 + i), bones=8, max_angle_deg=2.0)
        models.append(m)
    cam = Camera("camera", 640, 360)
    cam.render_normals = normals
    return W.Workload("flat", cam, Scene("flat", W._world(0.3)), W.icosphere_scene().lights, models)


@pytest.mark.gpu
@pytest.mark.parametrize("stage", [0, 1], ids=["host", "device"])
@pytest.mark.parametrize("mode,normals", [(A.EXEC_BATCHED, False), (A.EXEC_BATCHED, True), (A.EXEC_PLAIN, True)],
                         ids=["batched", "batched_normals", "plain"])
@pytest.mark.parametrize("counts", [[900] * 6, [5000, 1, 2049, 64, 1300]], ids=["small_pairs", "large_pairs"])
def test_lean_records(oracle, counts, mode, normals, stage):
    """Within a budget that the records of skinned flat-shaded meshes do not fit, the vertex pass runs twice and the
    frame is the same."""
    wl = _flat_shaded(counts, 3, normals)
    print("lean records", counts, mode, normals, stage, flush=True)
    want = oracle.render_workload(wl)
    ballast = LightVolume("ballast", (0, 0, 0), (80, 80, 80), (1, 1, 1))   # as large as the download's packed lists
    used = []
    for budget in (lambda: 0, lambda: used[0] - 1):
        with Context(0, budget()) as ctx:
            ctx.poison_outputs(0x7FC0DEAD)
            _prepared(ctx, wl)
            ctx.upload_volume(ballast)
            ctx.set_tuning(model_stage=stage)
            ctx.profile()
            ctx.profile_read()
            ctx.render_inputs(ctx.inputs(wl.camera, wl.scene, wl.lights, wl.models, mode))
            ctx.profile(False)
            prof = ctx.profile_read()
            used.append(ctx.memory_used)
            ctx._check(ctx.L.t3d_volume_free(ctx.ctx, ballast.handle))
            compare_frames(ctx.download(), want)
    assert used[1] < used[0]
    assert "k_pair" not in prof and prof["k_vertex"][1] == 2 * prof["k_cull"][1]


@pytest.mark.gpu
def test_lean_records_without_allocation():
    """A frame that t3d_render_noalloc counts as just fitting its static array and whose records would be over it."""
    from tests.test_zz_no_alloc import DeviceArrays, _hip, _max_vertices, _noalloc_frame
    wl = _flat_shaded([340000], 1)
    arrays = DeviceArrays(_hip(), _max_vertices(wl))
    with Context(0) as ctx:
        try:
            ref = ctx.render_workload(wl)
            print("lean records without allocation", ref.survivors, flush=True)
            pairs, c, d, i = _noalloc_frame(ctx, wl, arrays, ctx.new_frame(), A.EXEC_BATCHED)
            assert [p[:4] for p in pairs] == [p[:4] for p in ref.pairs] and ref.survivors > 0
            np.testing.assert_array_equal(c.view(np.uint32), ref.color.view(np.uint32))
            np.testing.assert_array_equal(d.view(np.uint32), ref.depth.view(np.uint32))
            np.testing.assert_array_equal(i, ref.indices)
        finally:
            arrays.free()


@pytest.mark.gpu
@pytest.mark.parametrize("jobs", [1, 3])
def test_jobs_take_what_they_are_admitted_with(oracle, jobs):
    """Skinned flat-shaded jobs on a server with a budget, alone and batched with static ones: their frames take no more
    memory than the jobs' estimates and the quarter that every buffer is larger."""
    wls = [_flat_shaded([30000 + k, 20000], 4 if k == 0 else 0) for k in range(jobs)]
    with Context(0) as ctx:
        for wl in wls:
            _prepared(ctx, wl)
        before = ctx.memory_used
        with Server(ctx, slots=1, max_batch_jobs=4, hbm_budget=1 << 30) as srv:
            ids = [srv.submit(wl.camera, wl.scene, wl.lights, wl.models) for wl in wls]
            srv.drain()
            taken, admitted = ctx.memory_used - before, sum(srv.info(j).admitted_bytes for j in ids)
            print("admitted", jobs, admitted, "taken", taken, flush=True)
            assert taken <= admitted + admitted // 4
            for wl, j in zip(wls, ids):
                compare_frames(srv.download(j), oracle.render_workload(wl))
                srv.release(j)
