"""Benchmark of the geometry path (Camera.Render: transform, skinning, lighting,
cull, 512-bin depth sort, ebiten vertex assembly) on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload mixed]

A step is one Camera.Render frame of the workload, in the batched form (one
launch chain for all render pairs), with all meshes, bone palettes and light
volumes resident in HBM before timing.
Prints one JSON line.
"""
import argparse
import json
import os
import platform
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0   # MI355X HBM3E
METRIC = "tris/sec (xform+light+cull+sort), % HBM peak; p99 frame latency vs plain"

WORKLOADS = {
    "mixed": ("mixed_512", "512 models, vertex counts log-uniform in [24, 65536] (grids and icospheres), "
              "128 skinned with 32-bone 4-influence armatures, ambient + 1 directional + 8 point lights, "
              "1920x1080, per-part 512-bin back-to-front sort"),
    "cubes": ("cubes_4096", "4,096 unit cubes in a 200^3 box, ambient + 1 directional + 8 point lights, 1920x1080"),
    "heightfield": ("heightfield_1024", "1024x1024 heightfield (2,093,058 triangles), camera inside the terrain, "
                    "16 point + 1 directional + 1 volume light"),
    "crowd": ("crowd_256", "256 characters sharing one 2,562-vertex mesh, each with its own 64-bone armature "
              "given as poses and playing one of 8 one-second clips (24 rotation keys per bone) at its own "
              "playhead: keyframe sampling and palettes on the device every frame; ambient + 1 directional + 4 "
              "point lights, 1920x1080"),
    "icosphere_ref": ("icosphere_ref_1272v", "the icosphere configuration on the reference's own generator, "
                      "NewIcosphereMesh(2): 1,272 vertices, 1,280 triangles, flat normals"),
    "icosphere": ("icosphere_642v", "642-vertex icosphere, 640x360, ambient + directional + point light"),
}


def log(*a):
    print("[bench]", *a, file=sys.stderr, flush=True)


def frame_bytes(prof, frames):
    """Algorithmic bytes per frame: mesh streams + indices + uniforms + outputs."""
    tot = 0
    for name, (ms, launches, b) in prof.items():
        tot += b
    return tot / max(frames, 1)


def measured_traffic(workload, kernel):
    """HBM bytes per launch of `kernel` from the committed rocprofv3 --pmc
    summary (FETCH_SIZE + WRITE_SIZE, scaled by the copy-kernel calibration),
    or None when no summary exists for this workload."""
    path = os.path.join(ROOT, "profiles", "traffic_%s.json" % workload)
    try:
        with open(path) as fh:
            d = json.load(fh)
        return d["kernels"][kernel]["hbm_bytes_per_launch"]
    except (OSError, KeyError, ValueError):
        return None


def cpu_model():
    """The host CPU's model name as lscpu prints it (else /proc/cpuinfo's)."""
    try:
        import subprocess
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
        for line in out.splitlines():
            if line.strip().startswith("Model name:"):
                return line.split(":", 1)[1].strip()
    except (OSError, subprocess.SubprocessError):
        pass
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return platform.processor() or platform.machine()


def cpu_baseline(wl, warmup=3, frames=20):
    """The oracle (single-threaded restatement of the reference CPU path) on
    whole frames of the same workload, pinned to one core: `warmup` untimed
    frames, then `frames` timed ones.
    Returns the per-frame seconds of the timed frames and the warm-up count."""
    from oracle.oracle import Oracle
    o = Oracle()
    for i, m in enumerate(wl.meshes):
        o.register_mesh(m, 1 + i)
    for i, v in enumerate(wl.volumes):
        o.register_volume(v, 100000 + i)
    saved = [v.handle for v in wl.volumes]
    for i, v in enumerate(wl.volumes):
        v.handle = 100000 + i
    anims = wl.animations
    saved_anim = [an.handle for an in anims]
    for i, an in enumerate(anims):
        an.handle = an.handle or 200000 + i
        o.register_animation(an, an.handle)
    affinity = os.sched_getaffinity(0)
    os.sched_setaffinity(0, {min(affinity)})
    try:
        for _ in range(warmup):
            o.render_seconds(wl.camera, wl.scene, wl.lights, wl.models)
        times = [o.render_seconds(wl.camera, wl.scene, wl.lights, wl.models) for _ in range(frames)]
        warm = warmup
    finally:
        os.sched_setaffinity(0, affinity)
    for v, h in zip(wl.volumes, saved):
        v.handle = h
    for an, h in zip(anims, saved_anim):
        an.handle = h
    o.close()
    return times, warm


class _JobInputs:
    """Descriptors of one serving job, assembled from per-model descriptors
    built once for the pool (a model's descriptor does not depend on the job)."""

    def __init__(self, camera, world, lights, model_descs):
        from tetra3d_amd import _abi as A
        import ctypes as C
        self.cam = camera.desc()
        self.world = world
        self.lights = (A.LightDesc * max(1, len(lights)))(*[l.desc() for l in lights])
        self.models = (A.ModelDesc * max(1, len(model_descs)))(*model_descs)
        self.render = A.RenderDesc()
        self.render.camera = C.pointer(self.cam)
        self.render.world = C.pointer(self.world)
        self.render.light_count = len(lights)
        self.render.lights = self.lights
        self.render.model_count = len(model_descs)
        self.render.models = self.models
        self.render.exec_mode = A.EXEC_BATCHED


def job_inputs(ctx, models, jobs, scene):
    keep, cache = [], {}
    world = scene.world.desc()
    out = []
    for j in jobs:
        descs = []
        for i in j.model_ids:
            i = int(i)
            if i not in cache:
                cache[i] = models[i].desc(ctx.mesh_handle(models[i].mesh), keep)
            descs.append(cache[i])
        out.append(_JobInputs(j.camera, world, j.lights, descs))
    for o in out:
        o.keep = keep          # arrays the cached model descriptors point into
    return out


def serving_pool(args):
    """The serving workload's pool and trace, generated with worker
    processes: called before this process first touches the GPU."""
    from tetra3d_amd import workloads as W
    t = time.perf_counter()
    models, jobs = W.serving_trace(pool_size=args.pool, jobs=args.jobs, rate_hz=args.rate,
                                   workers=min(16, os.cpu_count() or 1))
    log("serving trace generated in %.1fs" % (time.perf_counter() - t))
    return models, jobs


def serve_bench(args):
    out = serve_measure(args, *serving_pool(args), args.extra_rates, args.plain_jobs)
    print(json.dumps(out), flush=True)
    return 0


def serve_measure(args, models, jobs, extra_rates, plain_jobs):
    """Serving loop: a resident pool of mixed models, a Poisson job trace
    replayed at its arrival times against the server (continuous batching on
    several streams, admission by HBM budget); per-job latency is submit ->
    outputs complete in HBM.  The plain per-job path (one kernel chain per
    render pair, one job at a time) runs on a sample of the same jobs."""
    from tetra3d_amd import _abi as A
    from tetra3d_amd import workloads as W
    from tetra3d_amd.runtime import Context
    from tetra3d_amd.serving import Server

    t = time.perf_counter()
    scene = W.Scene("serving", W._world(0.2))
    pool_v = sum(m.mesh.vertex_count for m in models)
    pool_t = sum(m.mesh.triangle_count for m in models)
    log("serving pool: %d models, %d vertices, %d triangles; %d jobs at %.0f/s"
        % (len(models), pool_v, pool_t, len(jobs), args.rate))
    ctx = Context(0)
    t = time.perf_counter()
    for m in models:
        ctx.upload_mesh(m.mesh)
    resident = ctx.memory_used
    log("pool resident in HBM: %.2f GB (uploaded in %.1fs)" % (resident / 1e9, time.perf_counter() - t))
    t = time.perf_counter()
    inputs = job_inputs(ctx, models, jobs, scene)
    job_tris = [sum(models[i].mesh.triangle_count for i in j.model_ids) for j in jobs]
    log("descriptors built in %.1fs; mean %.3g triangles per job" % (time.perf_counter() - t, np.mean(job_tris)))

    budget = int(args.serve_budget_gb * 1e9)
    with Server(ctx, slots=args.slots, max_batch_jobs=args.max_batch_jobs, hbm_budget=budget,
                auto_release=True) as srv:
        # warm-up: bursts of queued jobs form full-size batches on every slot,
        # so each pooled frame reaches its final size before timing
        warm = []
        for _ in range(3):
            warm += [srv.submit_inputs(inputs[k % len(inputs)]) for k in range(min(len(inputs), 16 * args.slots))]
            srv.drain()
        srv.reset_stats()
        # replay the trace at its arrival times
        arrivals = np.array([j.arrival_s for j in jobs]) - jobs[0].arrival_s
        t0 = time.perf_counter()
        for k, inp in enumerate(inputs):
            while time.perf_counter() - t0 < arrivals[k]:
                pass
            srv.submit_inputs(inp)
        srv.drain(timeout_ms=600000)
        wall = time.perf_counter() - t0
        st = srv.stats()
        del warm
        # latency under heavier load: the same trace replayed faster
        sweep = []
        for rate in [float(r) for r in extra_rates.split(",") if r]:
            srv.reset_stats()
            arr = arrivals * (args.rate / rate)
            t0 = time.perf_counter()
            for k, inp in enumerate(inputs):
                while time.perf_counter() - t0 < arr[k]:
                    pass
                srv.submit_inputs(inp)
            srv.drain(timeout_ms=600000)
            sw = srv.stats()
            sweep.append({"rate_hz": rate, "offered_tris_per_s": float(np.mean(job_tris)) * rate,
                          "value": sw.triangles / ((sw.last_done_ms - sw.first_submit_ms) / 1e3),
                          "p50_ms": sw.p50_ms, "p99_ms": sw.p99_ms, "batches": sw.batches})
            log("rate %.0f/s: %.3g tris/s, p50 %.3f p99 %.3f ms, %d batches"
                % (rate, sweep[-1]["value"], sw.p50_ms, sw.p99_ms, sw.batches))
        # capacity: the same jobs submitted all at once (closed loop)
        srv.reset_stats()
        for inp in inputs:
            srv.submit_inputs(inp)
        srv.drain(timeout_ms=600000)
        sat = srv.stats()
    span_s = (st.last_done_ms - st.first_submit_ms) / 1e3
    served = st.triangles / span_s
    mean_batch = st.completed / max(st.batches, 1)
    log("served %d jobs in %d batches (mean %.1f jobs/batch), %.3g tris/s, p50 %.3f p99 %.3f ms"
        % (st.completed, st.batches, mean_batch, served, st.p50_ms, st.p99_ms))
    capacity = sat.triangles / ((sat.last_done_ms - sat.first_submit_ms) / 1e3)
    log("saturated: %d jobs in %d batches, %.3g tris/s" % (sat.completed, sat.batches, capacity))

    # plain per-job path on a sample: one kernel chain per render pair, jobs one after another
    sample = list(range(0, len(jobs), max(1, len(jobs) // plain_jobs)))[:plain_jobs]
    ctx.render(jobs[sample[0]].camera, scene, jobs[sample[0]].lights,
               [models[i] for i in jobs[sample[0]].model_ids], A.EXEC_PLAIN, download=False)
    lat, tt = [], 0
    t0 = time.perf_counter()
    for k in sample:
        a = time.perf_counter()
        ctx.render(jobs[k].camera, scene, jobs[k].lights, [models[i] for i in jobs[k].model_ids], A.EXEC_PLAIN,
                   download=False)
        lat.append((time.perf_counter() - a) * 1e3)
        tt += job_tris[k]
    plain_value = tt / (time.perf_counter() - t0)
    log("plain per-job: %.3g tris/s, p50 %.3f ms per job" % (plain_value, np.percentile(lat, 50)))

    out = {
        "metric": "serving tris/sec with p50/p99 job latency (continuous batching vs plain per-job path)",
        "value": served,
        "unit": "tris/s",
        "n_gpus": 1,
        "higher_is_better": True,
        "dtype": "f32",
        "data": "synthetic (seeded SplitMix64 pool and Poisson trace, seed 0x7e7a3d)",
        "config": {"workload": "serving_pool%d" % args.pool, "pool_models": len(models), "pool_vertices": pool_v,
                   "pool_triangles": pool_t, "resident_bytes": resident, "jobs": len(jobs), "rate_hz": args.rate,
                   "offered_tris_per_s": float(np.mean(job_tris)) * args.rate, "slots": args.slots,
                   "max_batch_jobs": args.max_batch_jobs, "hbm_budget_bytes": budget},
        "latency_ms": {"p50": st.p50_ms, "p99": st.p99_ms,
                       "note": "Poisson arrivals at rate_hz; submit -> outputs complete in HBM, queueing included"},
        "batches": st.batches, "mean_jobs_per_batch": mean_batch, "completed": st.completed,
        "rejected": st.rejected, "wall_s": wall,
        "saturated": {"value": capacity, "batches": sat.batches, "p50_ms": sat.p50_ms, "p99_ms": sat.p99_ms,
                      "note": "all jobs submitted at once: the server's capacity"},
        "load_sweep": sweep,
        "plain": {"value": plain_value, "jobs_sampled": len(sample), "p50_ms": float(np.percentile(lat, 50)),
                  "p99_ms": float(np.percentile(lat, 99)), "speedup_served_vs_plain": served / plain_value,
                  "speedup_capacity_vs_plain": capacity / plain_value,
                  "speedup_at_rates_vs_plain": {str(int(x["rate_hz"])): x["value"] / plain_value for x in sweep}},
    }
    ctx.close()
    return out


def hbm_probe(nbytes=1 << 30, reps=20):
    """Practical HBM ceilings of this part: a 1 GiB fill, zero and copy
    (torch kernels, timed with events on the current stream), in GB/s of bytes
    moved (a copy counts its read and its write)."""
    import torch
    a = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    b = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    out = {}
    for name, fn, moved in [("fill", lambda: a.fill_(1), nbytes), ("zero", lambda: a.zero_(), nbytes),
                            ("copy", lambda: b.copy_(a), 2 * nbytes)]:
        fn()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(reps):
            fn()
        e1.record()
        torch.cuda.synchronize()
        ms = e0.elapsed_time(e1) / reps
        out[name] = {"ms": ms, "GBps": moved / (ms / 1e3) / 1e9}
        log("%s: %.3f ms, %.0f GB/s" % (name, ms, out[name]["GBps"]))
    print(json.dumps({"hbm_probe_bytes": nbytes, **out}), flush=True)
    return 0


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--workload", default="mixed", choices=sorted(WORKLOADS))
    ap.add_argument("--no-autotune", action="store_true")
    ap.add_argument("--tuning", default="", metavar="K=V,...",
                    help="launch shape to use instead of autotuning (fields of t3d_tuning), e.g. the config.tuning "
                         "of an earlier run, so profiler runs time the same shape")
    ap.add_argument("--plain-steps", type=int, default=3)
    ap.add_argument("--sync-only", action="store_true",
                    help="time synchronous frames only (no two frames in flight): for profiler runs, where "
                         "overlapping frames would stretch each dispatch")
    ap.add_argument("--cpu-warmup", type=int, default=3)
    ap.add_argument("--cpu-frames", type=int, default=20)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-serve-summary", action="store_true",
                    help="leave the serving summary (10,000-model pool, 2,000 jobs at 2,000/s) out of the frame line")
    ap.add_argument("--profile-steps", type=int, default=10)
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="BYTES",
                    help="only run the plain device copy of BYTES (counter calibration) and exit")
    ap.add_argument("--hbm-probe", action="store_true",
                    help="measure the HBM fill and copy ceilings (1 GiB, torch) instead of the frame benchmark")
    ap.add_argument("--serve", action="store_true", help="run the serving loop instead of the frame benchmark")
    ap.add_argument("--pool", type=int, default=10000)
    ap.add_argument("--jobs", type=int, default=2000)
    ap.add_argument("--rate", type=float, default=2000.0)
    ap.add_argument("--extra-rates", default="3000,4000,5000",
                    help="further Poisson rates (jobs/s) replayed after the headline one, for latency under load")
    ap.add_argument("--slots", type=int, default=4)
    ap.add_argument("--max-batch-jobs", type=int, default=32)
    ap.add_argument("--serve-budget-gb", type=float, default=24.0)
    ap.add_argument("--plain-jobs", type=int, default=20)
    args = ap.parse_args()

    if args.gpus != 1:
        print("bench.py: this build measures one GPU only (the geometry path runs on a single MI355X; "
              "multi-GPU sharding is a design note, not a measured configuration); got --gpus %d" % args.gpus,
              file=sys.stderr)
        return 2

    import ctypes as C

    from tetra3d_amd import _abi as A
    from tetra3d_amd import workloads as W
    from tetra3d_amd.runtime import Context

    if args.serve:
        return serve_bench(args)

    if args.hbm_probe:
        return hbm_probe()

    if args.copy_calibration:
        with Context(0) as ctx:
            ms = ctx.selftest_copy(args.copy_calibration, reps=20)
        print(json.dumps({"copy_bytes": args.copy_calibration, "kernel_ms": ms,
                          "GBps": 2 * args.copy_calibration / (ms / 1e3) / 1e9}), flush=True)
        return 0

    wname, wdesc = WORKLOADS[args.workload]
    # the serving summary's pool is generated first, by worker processes, before the GPU is touched
    serve_pool = None
    if args.workload == "mixed" and not args.no_serve_summary:
        serve_pool = serving_pool(args)
    t = time.perf_counter()
    wl = W.SCENES[args.workload]()
    log("workload %s: %d models, %d vertices, %d triangles (generated in %.1fs)"
        % (wname, len(wl.models), wl.vertex_count, wl.triangle_count, time.perf_counter() - t))

    ctx = Context(0)
    ctx.prepare(wl)
    inp = ctx.inputs(wl.camera, wl.scene, wl.lights, wl.models, A.EXEC_BATCHED)
    tuning = None
    if args.tuning:
        kv = dict(item.split("=") for item in args.tuning.split(",") if item)
        ctx.set_tuning(**{k: int(v) for k, v in kv.items()})
        tu = ctx.tuning()
        tuning = {f: getattr(tu, f) for f, _ in A.Tuning._fields_}
        log("tuning set to %s" % tuning)
    elif not args.no_autotune:
        t = time.perf_counter()
        tu = ctx.autotune(inp, reps=5)
        tuning = {f: getattr(tu, f) for f, _ in A.Tuning._fields_}
        log("autotune picked %s in %.1fs" % (tuning, time.perf_counter() - t))

    for _ in range(args.warmup):
        ctx.render_inputs(inp)
    pairs = ctx.pairs()
    survivors = int(sum(p[3] for p in pairs))
    tris = wl.triangle_count
    log("pairs %d, survivors %d of %d triangles" % (len(pairs), survivors, tris))

    # latency: K synchronous frames, each submit -> outputs complete in HBM
    per = []
    t0 = time.perf_counter()
    for _ in range(args.steps):
        a = time.perf_counter()
        ctx.render_inputs(inp)       # synchronous: returns when the frame's outputs are in HBM
        per.append((time.perf_counter() - a) * 1e3)
    t1 = time.perf_counter()
    sync_ms = (t1 - t0) * 1e3 / args.steps
    p50, p99 = float(np.percentile(per, 50)), float(np.percentile(per, 99))
    log("batched, synchronous: %.3f ms/frame, %.3g tris/s, p50 %.3f p99 %.3f ms"
        % (sync_ms, tris / (sync_ms / 1e3), p50, p99))

    # the same with the frame's outputs copied to pinned host memory (+D2H)
    try:
        hip = C.CDLL("libamdhip64.so.7")          # the HIP runtime the library already loaded
    except OSError:
        hip = C.CDLL("/opt/rocm/lib/libamdhip64.so")
    nv = 3 * survivors
    pinned = [C.c_void_p() for _ in range(3)]
    for ptr, nb in zip(pinned, (48, 48, 4)):
        if hip.hipHostMalloc(C.byref(ptr), C.c_size_t(max(1, nv * nb)), C.c_uint(0)) != 0:
            raise RuntimeError("hipHostMalloc of %d bytes failed" % (nv * nb))
    VP = C.POINTER(A.Vertex)
    per_d2h = []
    try:
        for k in range(args.warmup + args.steps):    # the first download grows the frame's packing buffer: untimed
            a = time.perf_counter()
            ctx.render_inputs(inp)
            ctx._check(ctx.L.t3d_frame_download(ctx.ctx, ctx.frame, C.cast(pinned[0], VP), C.cast(pinned[1], VP),
                                                C.cast(pinned[2], C.POINTER(C.c_uint32))))
            if k >= args.warmup:
                per_d2h.append((time.perf_counter() - a) * 1e3)
    finally:
        for ptr in pinned:
            hip.hipHostFree(ptr)
    d2h50, d2h99 = float(np.percentile(per_d2h, 50)), float(np.percentile(per_d2h, 99))
    log("batched, synchronous + D2H to pinned host: p50 %.3f p99 %.3f ms" % (d2h50, d2h99))

    # the raster sink: the frame drawn into the camera's textures on the device (t3d_frame_rasterize) and the
    # colour image copied to pinned host memory, what a host that shows the frame waits for
    img_bytes = 4 * wl.camera.width * wl.camera.height
    pimg = C.c_void_p()
    if hip.hipHostMalloc(C.byref(pimg), C.c_size_t(img_bytes), C.c_uint(0)) != 0:
        raise RuntimeError("hipHostMalloc of %d bytes failed" % img_bytes)
    per_img, per_rast = [], []
    try:
        for k in range(args.warmup + args.steps):    # the first draw sizes the sink's working buffers: untimed
            a = time.perf_counter()
            ctx.render_inputs(inp)
            b = time.perf_counter()
            ctx.rasterize()
            c = time.perf_counter()
            ctx._check(ctx.L.t3d_frame_download_images(ctx.ctx, ctx.frame, C.cast(pimg, C.POINTER(C.c_uint8)), None))
            if k >= args.warmup:
                per_img.append((time.perf_counter() - a) * 1e3)
                per_rast.append((c - b) * 1e3)
    finally:
        hip.hipHostFree(pimg)
    img50, img99 = float(np.percentile(per_img, 50)), float(np.percentile(per_img, 99))
    rast50 = float(np.percentile(per_rast, 50))
    log("batched, synchronous + raster sink + colour image to pinned host: p50 %.3f p99 %.3f ms (rasterize %.3f ms)"
        % (img50, img99, rast50))

    # throughput (the timed region): K frames submitted asynchronously into
    # two alternating frames, so frame k's host prologue overlaps frame k-1's
    # kernels; every frame's outputs are complete in HBM before the clock stops
    if args.sync_only:
        # profiler runs: every kernel runs alone, so per-dispatch durations
        # match the HIP-event timings below
        ms = sync_ms
    else:
        frames = [ctx.frame, ctx.new_frame()]
        for k in range(max(2, args.warmup)):
            ctx.render_async(inp, frames[k % 2])
        for f in frames:
            ctx.wait(f)
        t0 = time.perf_counter()
        for k in range(args.steps):
            ctx.render_async(inp, frames[k % 2])   # waits for frame k-2 of the same buffers first
        for f in frames:
            ctx.wait(f)
        t1 = time.perf_counter()
        ms = (t1 - t0) * 1e3 / args.steps
    value = tris / (ms / 1e3)
    log("batched, %s: %.3f ms/frame, %.3g tris/s" % ("synchronous" if args.sync_only else "pipelined", ms, value))

    # per-kernel durations with HIP events on the library's stream
    ctx.profile(True)
    ctx.profile_read(reset=True)
    for _ in range(args.profile_steps):
        ctx.render_inputs(inp)
    prof = ctx.profile_read(reset=True)
    ctx.profile(False)
    host_ms = prof.pop("host:prologue", (0.0, 1, 0))[0] / args.profile_steps
    host_uniforms_ms = prof.pop("host:pairs+uniforms", (0.0, 1, 0))[0] / args.profile_steps
    host_pair_list_ms = prof.pop("host:pair-list", (0.0, 1, 0))[0] / args.profile_steps
    host_pair_sort_ms = prof.pop("host:pair-sort", (0.0, 1, 0))[0] / args.profile_steps
    kern = {k: {"avg_ms": v[0] / max(v[1], 1), "launches_per_frame": v[1] / args.profile_steps,
                "algorithmic_bytes_per_launch": v[2] / max(v[1], 1)} for k, v in prof.items()}
    # the roofline is quoted for the longest kernel that moves algorithmic
    # bytes; sort scratch passes (histogram, scan, scatter) and the uniform
    # stage carry none, so their share shows in "kernels" instead
    frame_ms = lambda k: kern[k]["avg_ms"] * kern[k]["launches_per_frame"]
    longest = max(kern, key=frame_ms)
    dom = max((k for k in kern if kern[k]["algorithmic_bytes_per_launch"] > 0), key=frame_ms, default=longest)
    dk = kern[dom]
    achieved = dk["algorithmic_bytes_per_launch"] / (dk["avg_ms"] / 1e3) / 1e9
    B = frame_bytes(prof, args.profile_steps)
    device_ms = sum(v[0] for v in prof.values()) / args.profile_steps
    log("kernels: " + ", ".join("%s %.3fms" % (k, v["avg_ms"]) for k, v in sorted(kern.items())))

    # plain per-pair form of the same frame (one kernel chain per render pair)
    plain = None
    if args.plain_steps > 0:
        pinp = ctx.inputs(wl.camera, wl.scene, wl.lights, wl.models, A.EXEC_PLAIN)
        ctx.render_inputs(pinp)
        pper = []
        for _ in range(args.plain_steps):
            a = time.perf_counter()
            ctx.render_inputs(pinp)
            pper.append((time.perf_counter() - a) * 1e3)
        plain_ms = float(np.mean(pper))
        plain_value = tris / (plain_ms / 1e3)
        plain = {"value": plain_value, "ms_per_step": plain_ms, "p99_ms": float(np.percentile(pper, 99)),
                 "speedup_batched_vs_plain": value / plain_value}
        log("plain: %.3f ms/frame, %.3g tris/s" % (plain_ms, plain_value))

    serving = None
    if serve_pool is not None:
        full = serve_measure(args, *serve_pool, "", min(args.plain_jobs, 10))
        serve_pool = None
        serving = {"workload": full["config"]["workload"], "value": full["value"], "unit": "tris/s",
                   "p50_ms": full["latency_ms"]["p50"], "p99_ms": full["latency_ms"]["p99"],
                   "capacity_tris_per_s": full["saturated"]["value"], "capacity_p99_ms": full["saturated"]["p99_ms"],
                   "mean_jobs_per_batch": full["mean_jobs_per_batch"], "batches": full["batches"],
                   "completed": full["completed"], "offered_tris_per_s": full["config"]["offered_tris_per_s"],
                   "plain_per_job_tris_per_s": full["plain"]["value"],
                   "speedup_served_vs_plain": full["plain"]["speedup_served_vs_plain"],
                   "speedup_capacity_vs_plain": full["plain"]["speedup_capacity_vs_plain"],
                   "note": "10,000-model pool resident in HBM; 2,000 Poisson jobs at 2,000/s replayed at their arrival "
                           "times, 4 slots, up to 32 jobs per batch; latency submit -> outputs in HBM; capacity: the "
                           "same jobs submitted at once"}

    cpu = None
    if not args.no_cpu:
        times, warm = cpu_baseline(wl, args.cpu_warmup, args.cpu_frames)
        frames, el = len(times), float(sum(times))
        cpu = {"value": tris * frames / el, "unit": "tris/s", "cores": 1, "kind": "port",
               "sample": "%d warm-up and %d timed whole frame(s) of %s on the oracle (C restatement of camera.go/"
                         "model.go/light.go/sortingTriangles.go), single-threaded, pinned to one core, %.1f s timed"
                         % (warm, frames, wname, el),
               "frame_ms_median": 1e3 * float(np.median(times)), "frame_ms_p99": 1e3 * float(np.percentile(times, 99)),
               "host_cpu": cpu_model(), "nproc": os.cpu_count()}
        log("cpu baseline: %.3g tris/s (%d frames in %.1fs, median %.1f ms)"
            % (cpu["value"], frames, el, cpu["frame_ms_median"]))

    out = {
        "metric": METRIC,
        "value": value,
        "unit": "tris/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic (seeded SplitMix64 scene, seed 0x7e7a3d)",
        "config": {"workload": wname, "description": wdesc, "triangles_per_frame": tris,
                   "vertices_per_frame": wl.vertex_count, "render_pairs": len(pairs), "drawn_triangles": survivors,
                   "exec": "batched, two frames in flight", "tuning": tuning},
        "latency_ms": {"p50": p50, "p99": p99, "mean": sync_ms,
                       "note": "synchronous frames: submit -> outputs complete in HBM",
                       "with_d2h_p50": d2h50, "with_d2h_p99": d2h99,
                       "with_d2h_note": "submit -> outputs copied to pinned host memory (t3d_frame_download: "
                                        "survivors packed on the device, one copy per stream)",
                       "raster_image_p50": img50, "raster_image_p99": img99, "rasterize_p50": rast50,
                       "raster_image_note": "submit -> flushes drawn into the camera's colour and depth textures on "
                                            "the device (t3d_frame_rasterize) -> colour image (%d bytes) copied to "
                                            "pinned host memory" % img_bytes},
        "pipelined": None if args.sync_only else {"ms_per_step": ms, "frames_in_flight": 2},
        "hbm": {"algorithmic_bytes_per_frame": B, "frame_pct_of_peak": 100.0 * B / (ms / 1e3) / (HBM_PEAK_GBS * 1e9),
                "device_ms_per_frame": device_ms, "host_prologue_ms": host_ms,
                "host_pairs_uniforms_ms": host_uniforms_ms, "host_pair_list_ms": host_pair_list_ms,
                "host_pair_sort_ms": host_pair_sort_ms,
                "device_pct_of_peak": 100.0 * B / (device_ms / 1e3) / (HBM_PEAK_GBS * 1e9)},
        "plain": plain,
        "kernels": kern,
        "roofline": {"kernel": dom, "bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": measured_traffic(wname, dom),
                     "algorithmic_bytes_per_launch": dk["algorithmic_bytes_per_launch"], "avg_ms": dk["avg_ms"],
                     "longest_kernel": longest},
        "cpu_baseline": cpu,
        "serving": serving,
    }
    print(json.dumps(out), flush=True)
    ctx.close()
    return 0


if __name__ == "__main__":
    sys.exit(main())
