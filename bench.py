#!/usr/bin/env python3
"""Throughput of the HIP renderer on the random-sphere workload, one GPU.

A step is one full render of the workload: 1920x1080 pixels, 64 samples per
pixel, max depth 16, over the seeded 22x22 random-sphere field (488 spheres;
80 % Lambertian, 15 % metal, 5 % glass, 3 large spheres, ground sphere) --
scene and paths are synthetic.  The scene is resident in HBM before the timed
region (uploaded once, like the reference's scene initialisation that
precedes its timed draw(), render.rs:137-150).

Prints one JSON line with Msamples/s (one sample = one camera path carrying 4
hero wavelengths), the roofline of the timed steps' kernel (k_paths, which runs
whole paths; vector-ALU bound when the scene sits in LDS, bound by node fetches
otherwise) and in it that of the traversal in renders whose bounces are separate
launches, timed with HIP events on the render stream (the only one for workloads
without a profile of k_paths), the CPU baseline (the
CPU oracle -- a C++ restatement of the reference's renderer -- timed on this
host's cores over a bounded slice of the same workload) and, nested as
`time_to_rmse`, the metric's second half: the wall time the guided method
needs to reach the plain method's RMSE on the dispersive-prism scene
(--no-prism leaves it out).
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

WORKLOADS = {
    "spheres": dict(scene="spheres", width=1920, height=1080, samples=64, max_depth=16, views=1, count_spp=64),
    "cornell": dict(scene="cornell", width=256, height=256, samples=16, max_depth=8, views=1, count_spp=16),
    # 1,003,520-triangle noise-displaced icosphere, 4 camera views in one batch
    "mesh": dict(scene="mesh", width=1920, height=1080, samples=256, max_depth=12, views=4, count_spp=8),
    # dispersive prism caustics: equal-RMSE time of the guided and the plain method
    "prism": dict(scene="prism", width=1024, height=1024, samples=512, max_depth=24, views=1, count_spp=0),
    # 64 seeded scenes of uneven size, resolution and sample count, guided, in one batch
    "batch64": dict(scene="uneven_batch", count=64, max_depth=12),
}
MFMA_FP16_PEAK_TFLOPS = 2500.0
# network FLOPs per evaluation: 2 x (64x64 x 3 hidden + 40x64 output) multiply-adds
GUIDE_FLOP = 2 * (64 * 64 * 3 + 40 * 64)
HBM_PEAK_GBS = 8000.0
TRACE_KERNELS = {0: "k_trace_simple", 1: "k_trace", 2: "k_trace_simple (ww)", 3: "k_trace_lds"}
RAY_STREAM_BYTES = 48  # per traced ray: queue index in/out (8), origin+direction (32), hit t+record (8)


def log(*a):
    print("[bench]", *a, file=sys.stderr, flush=True)


VALU_PEAK_TLANE = 256 * 4 * 16 * 2.4e9 / 1e12  # CUs x SIMDs x lanes x clock: fp32 lane operations per second


def profiled_counters(workload, kernel, target_paths):
    """per-launch VALU counters of the dominant kernel from the committed
    rocprofv3 pass of the same workload (profiles/counters.json), if it
    profiled the same kernel and pass size; else None"""
    try:
        with open(os.path.join(ROOT, "profiles", "counters.json")) as f:
            t = json.load(f)[workload]
    except (OSError, KeyError, ValueError):
        return None
    if not t["kernel"].startswith(kernel) or t.get("target_paths") != target_paths:
        return None
    return t


def measured_traffic(workload, kernel, target_paths):
    """HBM bytes per launch of the dominant kernel from the committed rocprofv3
    FETCH_SIZE and WRITE_SIZE passes of the same workload (profiles/traffic.json,
    each counter scaled by what it reads for a 1 GiB copy), if they profiled
    the same kernel; else None"""
    try:
        with open(os.path.join(ROOT, "profiles", "traffic.json")) as f:
            t = json.load(f)[workload]
    except (OSError, KeyError, ValueError):
        return None
    if not t["kernel"].startswith(kernel) or t.get("target_paths") != target_paths:
        return None
    return int(t["fetch_bytes_per_launch"] + t["write_bytes_per_launch"])


def profiled_shape(workload):
    """the launch shape (pass size, traversal kernel) of the committed counter
    (or else traffic) profile of this workload's dominant kernel, or None"""
    t = None
    for fn in ("counters.json", "traffic.json"):
        try:
            with open(os.path.join(ROOT, "profiles", fn)) as f:
                t = json.load(f)[workload]
            break
        except (OSError, KeyError, ValueError):
            continue
    if t is None:
        return None
    names = {v: k for k, v in TRACE_KERNELS.items()}
    base = t["kernel"].split("<")[0]
    kern = [k for n, k in names.items() if n == base]
    return {"target_paths": t["target_paths"], "trace_kernel": kern[0]} if kern else None


def paths_roofline(workload, samples, ms_per_step):
    """the whole-path kernel over a timed step (its launches and the summing of
    the samples, 1% of it), from the committed rocprofv3 passes of the same
    workload (profiles/counters.json and traffic.json, per sample); None if it
    has none"""
    try:
        with open(os.path.join(ROOT, "profiles", "counters.json")) as f:
            c = json.load(f)[workload + "_paths"]
        with open(os.path.join(ROOT, "profiles", "traffic.json")) as f:
            t = json.load(f)[workload + "_paths"]
    except (OSError, KeyError, ValueError):
        return None
    n = samples / c["samples_per_launch"]
    util = c["SQ_THREAD_CYCLES_VALU"] / (64.0 * c["SQ_ACTIVE_INST_VALU"])
    insts = c["SQ_INSTS_VALU"] * n
    ops = insts * 64.0 * util / (ms_per_step * 1e-3) / 1e12
    traffic = (t["fetch_bytes_per_launch"] + t["write_bytes_per_launch"]) * n
    gbs = traffic / (ms_per_step * 1e-3) / 1e9
    valu = ops / VALU_PEAK_TLANE > gbs / HBM_PEAK_GBS
    ach, peak, unit = (ops, VALU_PEAK_TLANE, "T lane-op/s") if valu else (gbs, HBM_PEAK_GBS, "GB/s")
    return {"bound": "valu" if valu else "hbm", "achieved": round(ach, 3), "peak": peak, "unit": unit,
            "frac": round(ach / peak, 4), "kernel": "%s (whole paths)" % c["kernel"].split("<")[0],
            "traffic": int(traffic), "valu_insts_per_step": int(insts), "valu_utilization": round(util, 4),
            "valu_tlane_ops": round(ops, 3), "measured_gbs": round(gbs, 1),
            "note": "VALU instructions x 64 lanes x lane utilisation, or FETCH_SIZE + WRITE_SIZE bytes (between L2 and "
                    "the memory side, register spills and traversal stacks among them), of the profiled launches per "
                    "sample (profiles/counters.json, traffic.json) over the device time of a timed step"}


def view_jobs(sid, w, opts_fn):
    """the workload's jobs: view 0 with the scene camera, views 1.. with the
    other camera azimuths of the mesh scene"""
    from clovers_amd import abi, synth
    jobs = [(sid, opts_fn())]
    for v in range(1, w["views"]):
        cam = abi.camera_init(synth.MESH_VIEWS[v], (0.0, 1.0, 0.0), vertical_fov=40.0, aperture=0.0,
                              focus_distance=10.0)
        jobs.append((sid, opts_fn(), cam))
    return jobs


def cpu_baseline(scene, w, seconds):
    from clovers_amd import abi
    from oracle import py_oracle as po
    lib = None
    try:
        lib = po.lib(po.build(native=True))
        kind_note = "g++ -O3 -march=native"
    except Exception as e:  # no compiler on the host: use the shipped portable build
        log("native oracle build failed (%s); using the portable build" % e)
        lib = po.lib()
        kind_note = "g++ -O3 -march=x86-64-v3"
    threads = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    sc = po.OracleScene(scene, library=lib)
    opts = abi.render_opts(w["width"], w["height"], w["samples"], w["max_depth"], seed=1)
    # a central band growing outwards in slices of doubling height until about
    # `seconds` of CPU work are timed
    H = w["height"]
    lo = hi = H // 2
    dt, chunk = 0.0, 2
    while dt < seconds and (lo > 0 or hi < H):
        a = min(max(chunk // 2, 1), lo)
        b = min(chunk - a, H - hi)
        for r0, r1 in ((lo - a, lo), (hi, hi + b)):
            if r1 > r0:
                t0 = time.perf_counter()
                sc.render(opts, threads=threads, rows=(r0, r1))
                dt += time.perf_counter() - t0
        lo, hi, chunk = lo - a, hi + b, chunk * 2
    rows = hi - lo
    samples = rows * w["width"] * w["samples"]
    # a workload smaller than the budget is rendered again, with the next
    # sample indices, until it too is timed for about `seconds`
    reps = 1
    while dt < seconds and rows == H and reps < 1000:
        o2 = abi.render_opts(w["width"], w["height"], w["samples"], w["max_depth"], seed=1,
                             sample_offset=reps * w["samples"])
        t0 = time.perf_counter()
        sc.render(o2, threads=threads)
        dt += time.perf_counter() - t0
        samples += H * w["width"] * w["samples"]
        reps += 1
    what = ("%d renders of the whole %dx%d image" % (reps, w["width"], w["height"]) if reps > 1
            else "%d central rows of %dx%d" % (rows, w["width"], w["height"]))
    return {"value": samples / dt / 1e6, "unit": "Msamples/s", "cores": threads, "kind": "port",
            "sample": "%s at %d spp, depth %d (%d samples, %.1f s); CPU oracle = C++ restatement of the "
                      "reference renderer (%s, %d threads over rows)"
                      % (what, w["samples"], w["max_depth"], samples, dt, kind_note, threads)}


def time_to_rmse(curve, target):
    """device ms at which an RMSE-vs-time curve [(ms, rmse)] first reaches
    `target`: log-log interpolation between points, or an extrapolation
    from the last point with RMSE ~ t^-1/2 if it never does"""
    import math
    prev = None
    for t, e in curve:
        if e <= target:
            if prev is None:
                return t * (e / target) ** 2, False
            (t0, e0), (t1, e1) = prev, (t, e)
            if e0 == e1:
                return t1, False
            a = (math.log(target) - math.log(e0)) / (math.log(e1) - math.log(e0))
            return math.exp(math.log(t0) + a * (math.log(t1) - math.log(t0))), False
        prev = (t, e)
    t, e = curve[-1]
    return t * (e / target) ** 2, True


def prism_time_to_rmse(args):
    """Time-to-RMSE of guided vs plain rendering on the dispersive-prism scene:
    both methods render independent images at growing sample counts (each
    guided render trains its network from scratch, its training time
    included), the RMSE of luminance against a float64-accumulated plain
    reference is taken per image (the reference's own Monte Carlo variance,
    from its second moments, taken out of the mean squared error), and the
    device time the guided method needs to reach the plain method's RMSE at
    its largest sample count is read off the guided curve.  Returns a dict of
    the measurement."""
    import numpy as np

    import clovers_amd
    from clovers_amd import abi, synth
    w = dict(WORKLOADS["prism"])
    W, H, D = w["width"], w["height"], w["max_depth"]
    top = args.spp or args.prism_spp
    plain_spps = [s for s in (64, 128, 256, 512, 1024, 2048, 4096, 8192) if s <= top]
    guided_spps = [s for s in (32, 64, 128, 256, 512, 1024, 2048) if s <= max(top // 2, 32)]
    r = clovers_amd.Renderer(0)
    sid = r.upload(synth.prism())
    tuning = r.autotune([(sid, abi.render_opts(W, H, plain_spps[-1], D, seed=1))])
    guide_tuning = {k: v for k, v in (("guide_alpha", args.guide_alpha), ("guide_rounds", args.guide_rounds),
                                      ("guide_train_spp", args.guide_train_spp), ("guide_lr", args.guide_lr),
                                      ("guide_records", args.guide_records), ("guide_warmup", args.guide_warmup),
                                      ("guide_photons", args.guide_photons),
                                      ("guide_pre_rounds", args.guide_pre_rounds),
                                      ("guide_gate_density", args.guide_gate_density))
                    if v is not None}
    r.set_tuning(use_graph=0, **guide_tuning)  # every render here is a different one: nothing to replay
    tuning = r.tuning()
    log("tuning: %s" % tuning)
    t0 = time.perf_counter()
    ref, ref_sq = r.render(sid, abi.render_opts(W, H, args.ref_spp, D, seed=99, fp64_accum=1), want_sq=True)
    refY = ref[..., 1].astype(np.float64)
    ref_var = float(np.mean(np.maximum(ref_sq[..., 1].astype(np.float64) - refY ** 2, 0.0)) / args.ref_spp)
    log("reference: %d spp in %.1f s (its own MSE %.3g)" % (args.ref_spp, time.perf_counter() - t0, ref_var))
    curves = {}
    for name, g, spps in (("plain", abi.GUIDE_OFF, plain_spps), ("guided", abi.GUIDE_ON, guided_spps)):
        # the tuner ran on the plain job; a tail launch (if it chose one) would leave guided vertices unguided
        r.set_tuning(tail_depth=tuning["tail_depth"] if g == abi.GUIDE_OFF else 0)
        pts = []
        for spp in spps:
            mse, ms = 0.0, 0.0
            seeds = tuple(range(7, 7 + args.seeds))
            for sd in seeds:
                img, _ = r.render(sid, abi.render_opts(W, H, spp, D, seed=sd, guiding=g))
                ms += r.counters()["render_ms"] / len(seeds)
                mse += (np.mean((img[..., 1].astype(np.float64) - refY) ** 2) - ref_var) / len(seeds)
            pts.append((round(ms, 3), float(np.sqrt(max(mse, 1e-30)))))
            log("%-6s %4d spp: %9.1f ms  RMSE %.5f" % (name, spp, ms, pts[-1][1]))
        curves[name] = pts
    t_plain, target = curves["plain"][-1]
    t_guided, extrapolated = time_to_rmse(curves["guided"], target)
    ratio = t_plain / t_guided
    # the same read-off at the plain method's 512-spp RMSE (a shorter render: the training's fixed cost weighs more)
    short = None
    if 512 in plain_spps and top > 512:
        t_p512, e_p512 = curves["plain"][plain_spps.index(512)]
        t_g512, x512 = time_to_rmse(curves["guided"], e_p512)
        short = {"plain_spp": 512, "target_rmse": e_p512, "plain_ms": t_p512, "guided_ms": round(t_g512, 3),
                 "guided_extrapolated": x512, "ratio": round(t_p512 / t_g512, 3)}
    # the network's MFMA roofline: evaluations x FLOPs over the inference kernels' device time
    r.render(sid, abi.render_opts(W, H, guided_spps[-1], D, seed=7, guiding=abi.GUIDE_ON, flags=abi.FLAG_TIME_KERNELS))
    cg = r.counters()
    achieved = cg["guide_queries"] * GUIDE_FLOP / (cg["guide_infer_ms"] * 1e-3) / 1e12 if cg["guide_infer_ms"] else 0.0
    r.close()
    # the plain GPU method's throughput on this scene
    plain_rate = W * H * plain_spps[-1] / (t_plain * 1e-3) / 1e6
    return {
        "metric": "time-to-RMSE vs oracle, guided vs plain", "value": round(ratio, 3),
        "unit": "x (plain device time / guided device time at equal RMSE)", "higher_is_better": True,
        "workload": "prism %dx%d depth%d" % (W, H, D), "reference_spp": args.ref_spp,
        "reference": "plain method, float64 accumulation; its Monte Carlo variance (from its second moments) is "
                     "taken out of every image's mean squared error", "target_rmse": target,
        "plain_spp": plain_spps, "guided_spp": guided_spps,
        "plain_ms_at_target": t_plain, "guided_ms_at_target": round(t_guided, 3),
        "guided_extrapolated": extrapolated, "at_plain_512spp": short,
        "curves_ms_rmse": curves, "seeds_per_point": args.seeds,
        "renders": 2 * len(spps) * args.seeds,
        "tuning": dict(tuning, trace_kernel=abi.TRACE_NAMES[tuning["trace_kernel"]]),
        "guide_roofline": {"bound": "mfma", "achieved": round(achieved, 2), "peak": MFMA_FP16_PEAK_TFLOPS,
                           "unit": "TFLOP/s", "frac": round(achieved / MFMA_FP16_PEAK_TFLOPS, 5),
                           "kernel": "network evaluation (fp16 MFMA)",
                           "evaluations": cg["guide_queries"], "flop_per_evaluation": GUIDE_FLOP,
                           "infer_ms": round(cg["guide_infer_ms"], 3), "train_ms": round(cg["guide_train_ms"], 3),
                           "train_records": cg["guide_records"], "train_rounds": cg["guide_rounds"],
                           "render_ms": round(cg["render_ms"], 3)},
        "plain_gpu_msamples_per_s": round(plain_rate, 1),
    }


def run_prism(args):
    """The time-to-RMSE measurement as its own JSON line, with the CPU
    reference on the same scene beside the plain GPU method."""
    from clovers_amd import synth
    m = prism_time_to_rmse(args)
    w = dict(WORKLOADS["prism"])
    cpu = None
    if not args.no_cpu_baseline:
        log("cpu baseline ...")
        cpu = cpu_baseline(synth.prism(), dict(w, samples=512), args.cpu_seconds)
        log("cpu baseline %.3f Msamples/s on %d threads" % (cpu["value"], cpu["cores"]))
    line = {
        "metric": m["metric"], "value": m["value"], "unit": m["unit"], "n_gpus": 1, "steps": m["renders"],
        "warmup": 0, "ms_per_step": m["guided_ms_at_target"], "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32 (network fp16 on MFMA, fp32 accumulate)", "data": "synthetic",
        "config": {k: v for k, v in m.items() if k not in ("metric", "value", "unit", "guide_roofline")},
        "roofline": dict(m["guide_roofline"], traffic=None),
        "cpu_baseline": cpu,
        "plain_gpu_over_cpu": round(m["plain_gpu_msamples_per_s"] / cpu["value"], 1) if cpu else None,
    }
    print(json.dumps(line), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--workload", default="spheres", choices=sorted(WORKLOADS))
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-autotune", action="store_true", help="keep the default launch shapes")
    ap.add_argument("--target-paths", type=int, default=0,
                    help="fix the pass size instead of autotuning (profiling the tuner's choice)")
    ap.add_argument("--trace-kernel", default="", choices=["", "simple", "persistent", "ww", "lds_cached"],
                    help="fix the traversal kernel instead of autotuning")
    ap.add_argument("--ref-spp", type=int, default=65536, help="prism workload: samples of the reference image")
    ap.add_argument("--no-prism", action="store_true",
                    help="default workload: leave out the prism time-to-RMSE measurement nested in the line")
    ap.add_argument("--seeds", type=int, default=8,
                    help="prism workload: independent renders per curve point (the error is dominated by rare "
                         "caustic paths, so one render's RMSE is noisy)")
    ap.add_argument("--prism-spp", type=int, default=2048,
                    help="prism time-to-RMSE: samples per pixel of the plain method's last curve point (its RMSE is "
                         "the target; the read-off at its 512-spp RMSE is reported beside it)")
    ap.add_argument("--guide-alpha", type=float, default=None, help="prism workload: override the guide's share")
    ap.add_argument("--guide-rounds", type=int, default=None, help="prism workload: override the training rounds")
    ap.add_argument("--guide-lr", type=float, default=None, help="prism workload: override the Adam learning rate")
    ap.add_argument("--guide-train-spp", type=int, default=None,
                    help="prism workload: override the samples per pixel between training rounds")
    ap.add_argument("--guide-records", type=int, default=None,
                    help="prism workload: override the training records per round (multiples of 16384)")
    ap.add_argument("--guide-warmup", type=int, default=None, choices=[0, 1],
                    help="prism workload: 1 = training rounds on warm-up samples outside the image")
    ap.add_argument("--guide-photons", type=int, default=None,
                    help="prism workload: override the light-traced training records per round")
    ap.add_argument("--guide-pre-rounds", type=int, default=None,
                    help="prism workload: override the light-traced rounds before the first pass")
    ap.add_argument("--guide-gate-density", type=float, default=None,
                    help="prism workload: override the guiding gate's density threshold (0 = no gate)")
    ap.add_argument("--spp", type=int, default=0,
                    help="override the workload's samples per pixel (profiling runs: per-launch figures do not "
                         "depend on it; the JSON line then names the reduced workload)")
    ap.add_argument("--builder", default="host", choices=["host", "device"],
                    help="scene BVH builder: host binned SAH or the GPU clustering build")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="before rendering, copy 1 GiB device-to-device 3 times (a plain copy kernel of known "
                         "size, so profiler byte counters can be scaled)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path (the work would shard by "
              "sample range with one all-reduce of the pixel sums at the end)", file=sys.stderr)
        sys.exit(2)

    if args.workload == "prism":
        run_prism(args)
        return

    import numpy as np

    import clovers_amd
    from clovers_amd import abi, synth

    if args.calibrate_copy:
        import torch
        a = torch.empty(1 << 28, dtype=torch.float32, device="cuda")
        b = torch.empty_like(a)
        for _ in range(3):
            b.copy_(a)
        torch.cuda.synchronize()
        log("calibration copy: 3 x %d bytes" % (a.numel() * 4))
        del a, b

    w = dict(WORKLOADS[args.workload])
    r = clovers_amd.Renderer(0)
    scene = None
    if args.workload == "batch64":
        # uneven batch: 64 seeded scenes of different size, resolution and samples, guided, one batch
        t0 = time.perf_counter()
        batch = synth.uneven_batch(w["count"], seed=1)
        log("generated %d scenes in %.1f s" % (len(batch), time.perf_counter() - t0))
        t0 = time.perf_counter()
        sids, build_ms = [], 0.0
        for sc, _, _, _ in batch:
            sids.append(r.upload(sc, builder=args.builder))
            build_ms += r.counters()["build_ms"]
        log("uploaded in %.1f s (%s builds %.1f s)" % (time.perf_counter() - t0, args.builder, build_ms / 1e3))

        def jobs_for(flags=0, count=False):
            return [(sid, abi.render_opts(side, side, max(1, spp // 16) if count else spp, w["max_depth"],
                                          seed=k + 1, guiding=abi.GUIDE_ON, flags=flags))
                    for k, (sid, (_, _, side, spp)) in enumerate(zip(sids, batch))]
        samples = sum(side * side * spp for _, _, side, spp in batch)
        wl_name = "uneven batch of %d scenes (%d-%d triangles, 0-200 spheres), %d-%d px a side, %d-%d spp, " \
                  "depth %d, guided" % (len(batch), min(b[1] for b in batch), max(b[1] for b in batch),
                                        min(b[2] for b in batch), max(b[2] for b in batch),
                                        min(b[3] for b in batch), max(b[3] for b in batch), w["max_depth"])
        wcfg = {"jobs": len(batch), "triangles": sum(b[1] for b in batch), "pixels": sum(b[2] ** 2 for b in batch),
                "max_depth": w["max_depth"], "guiding": True}
    else:
        if args.spp:
            w["samples"] = args.spp
            w["count_spp"] = min(w["count_spp"], args.spp)
        scene = getattr(synth, w["scene"])()
        log("workload", args.workload, w)
        t0 = time.perf_counter()
        sid = r.upload(scene, builder=args.builder)
        build_ms = r.counters()["build_ms"]
        log("scene upload %.1f ms (%s build %.1f ms)" % ((time.perf_counter() - t0) * 1e3, args.builder, build_ms))

        def jobs_for(flags=0, count=False):
            spp = w["count_spp"] if count else w["samples"]
            return view_jobs(sid, w, lambda: abi.render_opts(w["width"], w["height"], spp, w["max_depth"], seed=1,
                                                             flags=flags))
        samples = w["width"] * w["height"] * w["samples"] * w["views"]
        wl_name = "%s %dx%d %dspp depth%d%s" % (w["scene"], w["width"], w["height"], w["samples"], w["max_depth"],
                                                " x%d views" % w["views"] if w["views"] > 1 else "")
        wcfg = {"views": w["views"], "width": w["width"], "height": w["height"], "spp": w["samples"],
                "max_depth": w["max_depth"]}

    jobs = jobs_for()
    if args.target_paths or args.trace_kernel:
        fixed = {}
        if args.target_paths:
            fixed["target_paths"] = args.target_paths
        if args.trace_kernel:
            fixed["trace_kernel"] = {v: k for k, v in abi.TRACE_NAMES.items()}[args.trace_kernel]
        r.set_tuning(**fixed)
        args.no_autotune = True
    tuning, tune_ms = r.tuning(), 0.0
    if not args.no_autotune:
        t0 = time.perf_counter()
        tuning = r.autotune(jobs)
        tune_ms = (time.perf_counter() - t0) * 1e3
        log("autotune %.0f ms: %s" % (tune_ms, tuning))
    # setup, like the scene upload and the autotuner: the library captures a
    # repeated render as a hipGraph on its second identical call, so two
    # renders here leave every warmup and timed step a graph replay
    # the output arrays are allocated here and overwritten by every later
    # render, as a caller's framebuffers are; every step still reads its
    # results back into them
    outs = None
    for i in range(2):
        outs = r.render_batch(jobs, outs=outs)
    for i in range(args.warmup):
        r.render_batch(jobs, outs=outs)
        log("warmup %d done" % i)
    gpu_ms = []
    t0 = time.perf_counter()
    for i in range(args.steps):
        outs = r.render_batch(jobs, outs=outs)
        gpu_ms.append(r.counters()["render_ms"])
        log("step %d: %.1f ms device" % (i, gpu_ms[-1]))
    wall = time.perf_counter() - t0
    # value and ms_per_step: each render's device time (HIP events on the render
    # stream around its whole launch sequence), the scene and paths resident in
    # HBM; the wall clock also holds the copy of the image back into the
    # caller's host arrays over PCIe, reported beside it
    wall_ms_per_step = wall / args.steps * 1e3
    ms_per_step = float(np.mean(gpu_ms))
    value = samples / (ms_per_step / 1e3) / 1e6
    # The reference's estimator lets a NaN hero-only sample through (draw_cpu.rs:131-133; thin-film and
    # refraction take sqrt(1 - c^2) unclamped, thin_film.rs:45-48, materials.rs:194-200), so a head-on
    # hit on the thin-film mesh can leave a non-finite pixel there too; count them.
    nonfinite = int(sum((~np.isfinite(img)).any(axis=-1).sum() for img, _ in outs))
    log("non-finite pixels: %d" % nonfinite)

    # the traversal in launches of its own.  Its committed counter profile (profiles/) was
    # taken at one launch shape; the roofline renders use that shape, whatever
    # the autotuner picked for the timed steps, so per-launch counters and
    # per-launch times describe the same launches
    shape = profiled_shape(args.workload)
    tuned = r.tuning()
    if shape:
        r.set_tuning(target_paths=shape["target_paths"], trace_kernel=shape["trace_kernel"], tail_depth=0)
    # ... per-launch durations from HIP events ...
    r.render_batch(jobs_for(flags=abi.FLAG_TIME_KERNELS))
    ct = r.counters()
    avg_launch_ms = ct["extend_ms"] / ct["extend_launches"]
    rays_per_launch = ct["rays"] / ct["extend_launches"]
    log("traversal: %d launches, %.2f ms total, %.4f ms mean, %.0f rays per launch"
        % (ct["extend_launches"], ct["extend_ms"], avg_launch_ms, rays_per_launch))
    # ... and algorithmic bytes per ray from the counting traversal (the same
    # paths; for the mesh a prefix of the samples: the per-ray means converge)
    r.render_batch(jobs_for(flags=abi.FLAG_COUNT, count=True))
    cc = r.counters()
    roof_tuning = r.tuning()
    r.set_tuning(**tuned)
    per_ray = (cc["node_visits"] * cc["node_bytes"] + cc["prim_tests"] * cc["prim_bytes"]) / cc["rays"] \
        + RAY_STREAM_BYTES
    per_launch = per_ray * rays_per_launch
    achieved = per_launch / (avg_launch_ms * 1e-3) / 1e9
    log("rays %d (%.2f per sample), nodes/ray %.2f, prims/ray %.2f, %.1f B/ray"
        % (ct["rays"], ct["rays"] / samples, cc["node_visits"] / cc["rays"], cc["prim_tests"] / cc["rays"], per_ray))
    lds_note = ("for the sphere field the BVH (125 nodes, 16 KB) and spheres (16 KB) are served from LDS, so HBM traffic per "
                "launch is far below the algorithmic bytes and the kernel is issue/latency bound (VALUBusy, "
                "VALUUtilization in profiles/)") if args.workload != "mesh" else (
                "the mesh BVH (226k nodes, 29 MB) and triangles (80 MB) exceed the LDS window and L2; node and "
                "triangle fetches come from HBM / the MALL (FETCH_SIZE in profiles/)")
    if args.workload == "batch64":
        lds_note = ("the timed steps take node and primitive turns by majority, these one of each a lane; "
                    "per-ray figures from a counting render at 1/16 of each job's samples over all 64 scenes; "
                    "record bytes are those of the job with the most samples")
    kname = TRACE_KERNELS[roof_tuning["trace_kernel"]]
    traffic = measured_traffic(args.workload, kname, roof_tuning["target_paths"])
    hbm = {"algorithmic_bytes_per_launch": int(per_launch), "algorithmic_gbs": round(achieved, 1),
           "measured_bytes_per_launch": traffic,
           "measured_gbs": round(traffic / (avg_launch_ms * 1e-3) / 1e9, 1) if traffic else None,
           "measured_frac": round(traffic / (avg_launch_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4) if traffic else None}
    counters = profiled_counters(args.workload, kname, roof_tuning["target_paths"])
    common = {"traffic": traffic,
              "kernel": "%s (4-wide BVH traversal + primitive tests)" % kname,
              "mean_launch_ms": round(avg_launch_ms, 4),
              "per_ray": {"node_visits": round(cc["node_visits"] / cc["rays"], 3),
                          "prim_tests": round(cc["prim_tests"] / cc["rays"], 3),
                          "node_bytes": cc["node_bytes"], "prim_bytes": cc["prim_bytes"],
                          "stream_bytes": RAY_STREAM_BYTES},
              "rays_per_sample": round(ct["rays"] / samples, 4),
              "launch_shape": {"target_paths": roof_tuning["target_paths"],
                               "trace_kernel": abi.TRACE_NAMES[roof_tuning["trace_kernel"]]}}
    if traffic is not None and (traffic / (avg_launch_ms * 1e-3) / 1e9 < 0.5 * HBM_PEAK_GBS) and counters:
        # not memory-bound (the tree and records sit in LDS / L2): the bound is
        # the vector ALU -- active lane operations per second over the SIMDs'
        util = counters["SQ_THREAD_CYCLES_VALU"] / (64.0 * counters["SQ_ACTIVE_INST_VALU"])
        lane_ops = counters["SQ_INSTS_VALU"] * 64.0 * util
        ach = lane_ops / (avg_launch_ms * 1e-3) / 1e12
        roofline = dict({"bound": "valu", "achieved": round(ach, 3), "peak": VALU_PEAK_TLANE,
                         "unit": "T lane-op/s", "frac": round(ach / VALU_PEAK_TLANE, 4)}, **common)
        roofline.update({"valu_insts_per_launch": counters["SQ_INSTS_VALU"], "valu_utilization": round(util, 4),
                         "valu_busy": counters.get("valu_busy"), "hbm": hbm,
                         "note": "achieved = VALU instructions per launch x 64 lanes x lane utilisation "
                                 "(rocprofv3 SQ_INSTS_VALU, SQ_THREAD_CYCLES_VALU / (64 SQ_ACTIVE_INST_VALU), "
                                 "profiles/counters.json) over the launch time measured here; peak = 256 CUs x 4 "
                                 "SIMDs x 16 lanes x 2.4 GHz; hbm: algorithmic bytes (counted node visits x 128 B + "
                                 "primitive tests x record bytes + 48 B of ray stream per ray) and rocprofv3 "
                                 "FETCH_SIZE + WRITE_SIZE per launch (profiles/traffic.json); " + lds_note})
    else:
        measured = traffic / (avg_launch_ms * 1e-3) / 1e9 if traffic else None
        ach = measured if measured else achieved
        # without a counter profile only the algorithmic bytes are known; they count node and
        # record fetches that L2 and LDS serve, so they give no HBM fraction: null
        frac = ach / HBM_PEAK_GBS if measured else None
        roofline = dict({"bound": "hbm", "achieved": round(ach, 1), "peak": HBM_PEAK_GBS,
                         "unit": "GB/s", "frac": round(frac, 4) if frac is not None else None}, **common)
        roofline.update({"hbm": hbm,
                         "note": "achieved = rocprofv3 FETCH_SIZE + WRITE_SIZE per launch of the same workload and "
                                 "kernel (profiles/traffic.json) over the launch time measured here (when no profile "
                                 "matches: the algorithmic bytes, and frac null); hbm.algorithmic: counted node "
                                 "visits x 128 B + "
                                 "primitive tests x record bytes + 48 B of ray stream per ray; " + lds_note})
    r.close()
    # without guided jobs the LDS-cached traversal stands for whole paths in one launch
    whole = args.workload != "batch64" and tuning["trace_kernel"] == abi.TRACE_LDS_CACHED
    paths = paths_roofline(args.workload, samples, ms_per_step) if whole else None
    if paths:
        roofline = dict(paths, traversal=roofline)

    cpu = None
    if not args.no_cpu_baseline and scene is not None:
        log("cpu baseline ...")
        cpu = cpu_baseline(scene, w, args.cpu_seconds)
        log("cpu baseline %.3f Msamples/s on %d threads" % (cpu["value"], cpu["cores"]))

    prism = None
    if args.workload == "spheres" and not args.no_prism:
        log("prism time-to-RMSE ...")
        prism = prism_time_to_rmse(args)
        log("prism time-to-RMSE guided/plain %.3f" % prism["value"])

    line = {
        "metric": "Msamples/s at 1 GPU", "value": round(value, 3), "unit": "Msamples/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(ms_per_step, 3), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": dict({"workload": wl_name}, **wcfg, **{
                   "samples_per_step": samples, "nonfinite_pixels": nonfinite, "device_ms_per_step": round(ms_per_step, 3),
                   "wall_ms_per_step_with_readback": round(wall_ms_per_step, 3),
                   "wall_msamples_per_s_with_readback": round(samples / (wall_ms_per_step / 1e3) / 1e6, 3),
                   "parallelism": "1 GPU, %s" % ("whole paths in one launch" if whole else "wavefront"),
                   "scene_builder": args.builder, "scene_build_ms": round(build_ms, 1),
                   "tuning": dict(tuning, trace_kernel=abi.TRACE_NAMES[tuning["trace_kernel"]]),
                   "autotune_ms": round(tune_ms, 1)}),
        "roofline": roofline,
        "cpu_baseline": cpu,
        "gpu_over_cpu": round(value / cpu["value"], 1) if cpu else None,
        "time_to_rmse": prism,
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
