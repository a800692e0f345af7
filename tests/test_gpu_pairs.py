"""Frames of small render pairs, which one workgroup each draws whole: pairs at and one past the sizes where the
workgroup changes or the chain of passes takes over, static and skinned, in the three sort modes, built on the host and
on the device, against the oracle bit for bit."""
import numpy as np
import pytest

from tetra3d_amd import _abi as A
from tetra3d_amd import workloads as W
from tetra3d_amd.scene import Camera, Mesh, Model, Scene
from tests.parity import compare_frames

SIZES = [(3, 1, 1), (3, 2, 2), (128, 128, 3), (129, 128, 2), (128, 129, 2), (128, 100, 600), (300, 65, 600),
         (1024, 2048, 2), (1025, 2048, 2), (1024, 2049, 2), (63, 1023, 5), (2816, 5632, 64), (2817, 5632, 64)]


def _mesh(v, t, seed):
    """v points before the camera and t triangles between neighbours of them, three different ones each (the reference
    lights a corner that a triangle names twice two times)."""
    r = np.random.default_rng(seed)
    pos = np.stack([r.uniform(-3, 3, v), r.uniform(-2, 2, v), r.uniform(-14, 0.5, v)], axis=1)
    nrm = r.normal(size=(v, 3))
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    a = np.arange(t) * max(1, v // t) % v
    far = 20 + 3 * (np.arange(t) % 5) if v > 40 else 2
    idx = np.stack([a, (a + 1 + np.arange(t) // v) % v, (a + far) % v], axis=1)
    idx[-1] = [0, v // 2, v - 1]
    assert all(len(set(x)) == 3 for x in idx.tolist())
    return Mesh("m%d" % seed, pos, nrm, idx, colors=np.c_[r.random((v, 3)), np.ones(v)], uvs=r.random((v, 2)))


def _one_workgroup_each(v, t, count):
    return (v <= 1024 and t <= 2048) or (v <= 2816 and t <= 5632 and count >= 64)


@pytest.mark.gpu
@pytest.mark.parametrize("stage", [2, 1], ids=["host", "device"])
@pytest.mark.parametrize("visible", [True, False], ids=["culled", "all"])
@pytest.mark.parametrize("size", SIZES, ids=["v%d_t%d_x%d" % s for s in SIZES])
def test_pair_sizes(gpu_ctx, oracle, size, visible, stage):
    v, t, count = size
    r = np.random.default_rng(7)
    meshes = [_mesh(v, t, k) for k in range(min(count, 3))]
    models = []
    for i in range(count):
        m = Model("m%d" % i, meshes[i % len(meshes)])
        m.set_local_position(*r.uniform(-0.5, 0.5, 3))
        m.frustum_culling = False
        models.append(m)
    for k, mesh in enumerate(meshes):
        mesh.mesh_parts[0].material.triangle_sort_mode = [A.SORT_BACK_TO_FRONT, A.SORT_FRONT_TO_BACK, A.SORT_NONE][k]
        mesh.mesh_parts[0].material.backface_culling = k != 1
    if len(meshes) > 1:                       # one mesh in three skinned, each model with its own bones
        for i, m in enumerate(models):
            if i == 1:
                W._skin(m, W.SplitMix64(5), bones=8)
            elif i % len(meshes) == 1:
                m.skinned, m.bone_influences = True, models[1].bone_influences + np.float32(0.01 * (i % 7))
    cam = Camera("camera", 800, 450)
    cam.process_only_visible = visible
    wl = W.Workload("pairs", cam, Scene("pairs", W._world(0.2)), W.icosphere_scene().lights, models)
    print("pairs", size, visible, stage, flush=True)
    saved = gpu_ctx.tuning()
    gpu_ctx.set_tuning(model_stage=stage)
    try:
        gpu_ctx.profile(True)
        gpu_ctx.profile_read(reset=True)
        got = gpu_ctx.render_workload(wl)
        ran = gpu_ctx.profile_read(reset=True)
    finally:
        gpu_ctx.profile(False)
        gpu_ctx.L.t3d_set_tuning(gpu_ctx.ctx, saved)
    assert ("k_pair" in ran) == _one_workgroup_each(*size) != ("k_cull" in ran)
    assert ("k_models" in ran) == (stage == 1 and visible)     # without culling the host builds every frame
    s = compare_frames(got, oracle.render_workload(wl))
    if not visible:
        assert s["survivors"] == count * t
    elif t > 2:                               # some of each mesh's triangles lie behind the camera or face away
        assert 0 < s["survivors"] < count * t
