"""Frames in flight together overlap on the device: in a process of its own (whose streams are one context's, two
frames' and the null stream), two alternating frames take well under the time of waiting for each, in whichever order
the streams come to be."""
import os
import subprocess
import sys

import pytest

from tests.conftest import ROOT

CHILD = """
import sys, time
from tetra3d_amd import workloads as W
from tetra3d_amd.runtime import Context

if sys.argv[1] == "torch_first":
    import torch
    torch.zeros(4, device="cuda")
wl = W.heightfield_scene(n=357)
with Context(0) as ctx:
    if sys.argv[1] == "meshes_first":
        ctx.prepare(wl)
    frames = [ctx.frame, ctx.new_frame()]
    ctx.prepare(wl)
    inp = ctx.inputs(wl.camera, wl.scene, wl.lights, wl.models)

    def flight(n=50):
        t = time.perf_counter()
        for k in range(n):
            ctx.render_async(inp, frames[k % 2])
        for f in frames:
            ctx.wait(f)
        return (time.perf_counter() - t) / n * 1e6

    def alone(n=50):
        t = time.perf_counter()
        for k in range(n):
            ctx.render_inputs(inp)
        return (time.perf_counter() - t) / n * 1e6

    flight(), alone()
    print("in flight %.1f alone %.1f" % (min(flight() for _ in range(30)), min(alone() for _ in range(10))), flush=True)
"""


@pytest.mark.gpu
@pytest.mark.parametrize("order", ["frames_first", "meshes_first", "torch_first"])
def test_frames_overlap(order):
    """A 357 x 357 grid, measured: 0.55 of the time of waiting for each frame, 0.90 where the two frames' streams share a
    hardware queue."""
    r = subprocess.run([sys.executable, "-c", CHILD, order], cwd=ROOT, timeout=100, stdout=subprocess.PIPE,
                       env={**os.environ, "PYTHONPATH": ROOT})
    out = r.stdout.decode()
    print(order, out, flush=True)
    assert r.returncode == 0
    flight, alone = (float(x) for x in (out.split()[2], out.split()[4]))
    assert flight < 0.75 * alone
