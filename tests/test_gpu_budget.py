"""What a frame takes of its context's memory budget."""
import numpy as np
import pytest

from tetra3d_amd import _abi as A
from tetra3d_amd import workloads as W
from tetra3d_amd.runtime import Context
from tetra3d_amd.scene import Camera, Model, Scene
from tests.parity import compare_frames
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
