"""The assembly's split of a render pair's lists: pairs whose triangle counts lie at the edges of its wavefronts'
chunks, its blocks and the sort's tiles, one after another so that each starts at another offset from a 1 KB run of
the output, against the oracle bit for bit."""
import numpy as np
import pytest

from tetra3d_amd import _abi as A
from tetra3d_amd import workloads as W
from tetra3d_amd.scene import Camera, Mesh, Model, Scene
from tests.parity import compare_frames

COUNTS = [1, 2, 3, 7, 8, 9, 63, 64, 65, 71, 72, 127, 128, 129, 255, 256, 257, 263, 511, 512, 513, 1023, 2047, 2048, 2049,
          2304, 4097]


def _strip(n, name):
    """A mesh of n separate triangles in front of the camera, at depths that the sort reorders."""
    r = np.random.default_rng(n)
    at = np.stack([r.uniform(-2, 2, n), r.uniform(-1, 1, n), r.uniform(-12, -4, n)], axis=1)
    pos = (at[:, None, :] + r.uniform(-0.2, 0.2, (n, 3, 3))).reshape(-1, 3)
    nrm = np.tile([0, 0, 1], (3 * n, 1))
    colors = np.c_[r.random((3 * n, 3)), np.ones(3 * n)] if n % 2 else None
    return Mesh(name, pos, nrm, np.arange(3 * n).reshape(-1, 3), colors=colors, uvs=r.random((3 * n, 2)))


def _scene(counts, normals):
    models = []
    for i, n in enumerate(counts):
        m = Model("m%d" % i, _strip(n, "strip%d" % i))
        m.frustum_culling = False
        models.append(m)
    cam = Camera("camera", 640, 360)
    cam.process_only_visible = False           # every triangle is drawn: the counts are the survivors'
    cam.render_normals = normals
    return W.Workload("strips", cam, Scene("strips", W._world(0.3)), W.icosphere_scene().lights, models)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [A.EXEC_BATCHED, A.EXEC_PLAIN], ids=["batched", "plain"])
@pytest.mark.parametrize("normals", [False, True], ids=["lists", "normals"])
@pytest.mark.parametrize("tile,split", [(2048, 8), (2048, 1), (64, 1), (512, 8)])
def test_chunk_edges(gpu_ctx, oracle, tile, split, normals, mode):
    wl = _scene(COUNTS, normals)
    print("assembly edges", tile, split, normals, mode, flush=True)
    saved = gpu_ctx.tuning()
    gpu_ctx.set_tuning(triangle_tile=tile, assemble_split=split)
    try:
        g = gpu_ctx.render_workload(wl, exec_mode=mode)
    finally:
        gpu_ctx.L.t3d_set_tuning(gpu_ctx.ctx, saved)
    s = compare_frames(g, oracle.render_workload(wl))
    assert s["survivors"] == sum(COUNTS)


@pytest.mark.gpu
@pytest.mark.parametrize("normals", [False, True], ids=["lists", "normals"])
@pytest.mark.parametrize("counts", [[5], [12, 12, 12], [300, 40], [256, 257], [1, 2000]])
def test_small_pairs(gpu_ctx, oracle, counts, normals):
    """Frames whose largest pair is smaller than a tile: with normal lists the chain draws them, with fewer blocks per
    tile in its assembly (1, 1, 2, 2 and the full 8); without, one workgroup draws each pair (but for the last frame's,
    which are too large for that)."""
    wl = _scene(counts, normals)
    print("assembly small", counts, normals, flush=True)
    gpu_ctx.profile(True)
    try:
        gpu_ctx.profile_read(reset=True)
        got = gpu_ctx.render_workload(wl)
        ran = gpu_ctx.profile_read(reset=True)
    finally:
        gpu_ctx.profile(False)
    chain = normals or 3 * max(counts) > 2816
    assert ("k_assemble" in ran) == chain == ("k_pair" not in ran)
    s = compare_frames(got, oracle.render_workload(wl))
    assert s["survivors"] == sum(counts)
