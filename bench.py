"""Benchmark: Msamples/s of the GPU path tracer on one MI355X.

python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload NAME]

A step is one full render of the workload's image at its sample count,
inputs resident in HBM, output image in HBM.  Prints one JSON line.

Workloads:
  config1   icosphere(3) on a ground quad, sky cube map 6x64x64 with a
            sun disk, 256x256, 4 spp, 3 bounces, per-pixel PCG streams,
            the reference's estimator (ComputeRadianceForPath) -- the
            configuration whose CPU run is the reference's own workload.
  soup      closest hit only: 2^22 rays vs a 1M-triangle soup (Mrays/s).

The roofline entry is for the dominant kernel of the workload (the
closest-hit traversal, k_extend / k_closest_mesh): algorithmic bytes per
launch = per ray 24 (ray) + 20 (hit record) + 24 per slab test + 36 per
triangle test, the test counts taken from a counting run of the same
launches; divided by the mean launch time from HIP events on the launch
stream.  The cpu_baseline entry times the oracle (the C restatement of the
reference tracer) on a bounded sample of the same workload on this host.
"""
import argparse
import ctypes as C
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "Msamples/s at 1 GPU; time-to-relMSE 1e-3, guided vs plain GPU tracer"
HBM_PEAK_GBS = 8000.0
MFMA_FP16_PEAK_TFLOPS = 2500.0   # dense FP16 MFMA, MI355X
# Algorithmic bytes of the closest-hit walk, per unit: a ray's 24 bytes in
# and its hit record out (8 bytes, triangle and t, for the closest-hit
# kernel; 20 bytes, t, u, v, instance, triangle, for the path tracer's
# extension kernel); one box test = a full-precision box (24 bytes; the
# four-wide nodes store a child box in 6 quantized bytes plus a quarter of
# the node's 32-byte header, so the kernels fetch less than this); one
# triangle test = its three vertices (36 bytes); one instance entry = 128
# bytes (index, inverse and forward 3x4 rows, cull scale, mesh id and
# pointers).
RAY_BYTES, HIT_BYTES_MESH, HIT_BYTES_SCENE = 24, 8, 20
BOX_BYTES, TRI_BYTES, ENTRY_BYTES = 24, 36, 128
# HBM bytes per traced ray of the closest-hit kernel, measured with rocprofv3
# --pmc FETCH_SIZE and WRITE_SIZE per dispatch (FETCH scaled x2.0, WRITE
# x1.0 by the 1 GiB copy of `--workload copy` on the same box; config5: the
# plain tracer's launches, `--no-guided`); the roofline's "traffic" is this
# times the rays of one launch.
TRAFFIC_BYTES_PER_RAY = {"config5": 1.3923e9 / 2036866, "soup": 1.0627e9 / 4194304}
# What bounds the closest-hit kernel in fact, from counter runs of the same
# kernel and workload: the VALU issue rate and the texture path, not HBM.
# valu_busy: share of the SIMDs' cycles issuing VALU work (SQ_INSTS_VALU x 4 cycles per wave64
# instruction over 1024 SIMDs x the dispatches' mean duration x 2.4 GHz);
# valu_insts_per_ray: SQ_INSTS_VALU per traced ray.  The roofline "frac"
# prices the algorithmic bytes, "traffic_frac" the counter-measured ones.
LIMITER = {"config5": {"kind": "VALU issue and fetches", "valu_busy": 0.74,
                       "valu_insts_per_ray": 172,
                       "source": "profiles/hbm_traffic_config5_soup.md"}}
TRAFFIC_SOURCE = ("rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE of the same kernel and "
                  "workload (profiles/hbm_traffic_config5_soup.md), FETCH x2.0 and "
                  "WRITE x1.0 by a 1 GiB copy calibration")


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def host_cpu():
    """The host CPUs this process may use: the CPU model, the machine's
    logical CPU count (nproc), the CPUs in this process's affinity mask, the
    cgroup quota in CPUs where one is set, and the worker count the CPU
    baselines use -- the process's CPU share (OMP_NUM_THREADS where the
    host sets it, else the affinity mask), so a baseline never runs more
    threads than the cores it is given."""
    model = None
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    affinity = len(os.sched_getaffinity(0))
    quota = None
    try:
        with open("/sys/fs/cgroup/cpu.max") as f:
            q, period = f.read().split()
            if q != "max":
                quota = float(q) / float(period)
    except (OSError, ValueError):
        pass
    share = affinity
    if os.environ.get("OMP_NUM_THREADS", "").isdigit():
        share = min(share, int(os.environ["OMP_NUM_THREADS"]))
    if quota:
        share = min(share, max(1, int(quota)))
    return {"model": model, "nproc": os.cpu_count(), "affinity": affinity,
            "cgroup_cpus": quota, "threads": max(1, share)}


def cpu_baseline_config1(threads, spp=16):
    """The oracle's threaded tile renderer (64x64 tiles pulled from an atomic
    counter as src/main.cpp:731-844 does) on config 1 with the reference's
    own BVH and estimator, `spp` samples per pixel."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    from _libs import (SPO_EST_UNBIASED, SPO_HIT_REFERENCE, SPO_RNG_PCG,
                       SPO_TX_LIBM, SpoConfig, oracle)
    from _scenes import load_oracle
    from vk_cinematic_amd import scenes

    desc = scenes.config1(256, 256, env="cube")
    O = oracle()
    s, cam = load_oracle(desc)
    cfg = SpoConfig(rng=SPO_RNG_PCG, tx=SPO_TX_LIBM, hit=SPO_HIT_REFERENCE,
                    estimator=0, samplesPerPixel=spp, bounces=3, radianceClamp=10.0,
                    jitterYFirst=1, seed=0x5EED)
    px = np.zeros(256 * 256 * 4, np.float32)
    O.spo_render_threaded(s, C.byref(cam), C.byref(cfg), 64, 64, threads, px,
                          np.zeros(12, np.uint64))  # warm-up
    secs = []
    for _ in range(3):
        secs.append(O.spo_render_threaded(s, C.byref(cam), C.byref(cfg), 64, 64,
                                          threads, px, np.zeros(12, np.uint64)))
    O.spo_scene_destroy(s)
    sec = float(np.median(secs))
    return {"value": 256 * 256 * spp / sec / 1e6, "unit": "Msamples/s",
            "cores": threads, "kind": "port",
            "sample": f"config1 256x256, {spp} spp, 3 bounces, reference BVH and "
                      f"estimator, median of 3 after 1 warm-up ({sec:.2f} s each)"}


def cpu_baseline_soup(threads, tris, o, d, repeats=3):
    """The oracle's restatement of the closest-hit traversal (the binary SAH
    hierarchy of the same build), all host threads, on all 2^22 rays: one
    warm-up pass, then the median of `repeats` timed passes."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    from _libs import oracle
    import vk_cinematic_amd as V

    nodes, order, _ = V.bvh_build_host(tris)
    n = len(o)
    rays = np.ascontiguousarray(np.concatenate([o, d], 1).ravel())
    p = np.zeros(n, np.uint32)
    t = np.zeros(n, np.float32)
    O = oracle()
    nodes = np.ascontiguousarray(nodes.ravel())
    tris = np.ascontiguousarray(tris.ravel())
    secs = []
    for k in range(repeats + 1):
        t0 = time.perf_counter()
        O.spo_bvh2_closest(nodes, order, tris, rays, n, threads, p, t, None, None)
        if k:
            secs.append(time.perf_counter() - t0)
    sec = float(np.median(secs))
    return {"value": n / sec / 1e6, "unit": "Mrays/s", "cores": threads,
            "kind": "port",
            "sample": f"all {n} rays, same SAH build, median of {repeats} passes "
                      f"after a warm-up ({sec:.2f} s per pass)"}


def cpu_baseline_irradiance(sky, fw, fh):
    """The oracle's restatement of CreateIrradianceCubeMap (one host thread,
    double-evaluated transcendentals like the GPU line), the whole cube map."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    from _libs import oracle

    eh, ew = sky.shape[:2]
    out = np.zeros(6 * fw * fh * 4, np.float32)
    t0 = time.perf_counter()
    oracle().spo_create_irradiance_cubemap(np.ascontiguousarray(sky.ravel()), ew, eh,
                                           fw, fh, 10.0, 1, out)
    sec = time.perf_counter() - t0
    samples = 6 * fw * fh * 63 * 16
    return {"value": samples / sec / 1e9, "unit": "Gsamples/s", "cores": 1,
            "kind": "port",
            "sample": f"the whole {fw}x{fh} cube map ({sec:.2f} s)"}


def bench_config1(args, V, scenes):
    dev = V.Device(0)
    desc = scenes.config1(256, 256, env="cube")
    s, cam = scenes.load_gpu(dev, desc)
    tiles = V.ComputeTiles(256, 256, 64, 64)
    spp, bounces = 4, 3
    img = dev.alloc(256 * 256 * 16)
    ctx = V.make_context(cam, s, spp=spp, bounces=bounces, clamp=10.0,
                         estimator=V.EST_PARITY, rng=V.RNG_PCG, seed=0x5EED)
    for _ in range(args.warmup):
        V.path_trace_tiles_device(ctx, tiles, img)
    dev.synchronize()
    ext_ms, ext_n, tot_ms, steps_ms = 0.0, 0, 0.0, []
    t0 = time.perf_counter()
    for _ in range(args.steps):
        ts = time.perf_counter()
        V.path_trace_tiles_device(ctx, tiles, img)
        steps_ms.append((time.perf_counter() - ts) * 1e3)
        tim = dev.last_timings()
        ext_ms += tim["extend"][0]
        ext_n += tim["extend"][1]
        tot_ms += tim["total"][0]
    dev.synchronize()
    wall = time.perf_counter() - t0
    # counting run of the same launches: slab and triangle tests, rays
    cctx = V.make_context(cam, s, spp=spp, bounces=bounces, clamp=10.0,
                          estimator=V.EST_PARITY, rng=V.RNG_PCG, seed=0x5EED,
                          collect=True)
    m = V.path_trace_tiles_device(cctx, tiles, img)
    rays = m.values[V.METRIC_RAYS]
    box = m.values[V.METRIC_AABB_TESTS]
    tri = dev.last_counters()["tri_tests"]
    bytes_step = (RAY_BYTES + HIT_BYTES_SCENE) * rays + BOX_BYTES * box + TRI_BYTES * tri
    launches = ext_n / args.steps
    per_launch_bytes = bytes_step / launches
    mean_ms = ext_ms / ext_n
    achieved = per_launch_bytes / (mean_ms * 1e-3) / 1e9
    samples = 256 * 256 * spp
    res = {
        "metric": METRIC,
        "value": samples * args.steps / wall / 1e6,
        "unit": "Msamples/s",
        "ms_per_step": wall * 1e3 / args.steps,
        "dtype": "f32",
        "config": {"workload": "config1: icosphere(3) + 20x20 ground quad, sky cube "
                               "6x64x64 (sun 50), 256x256, 4 spp, 3 bounces, "
                               "parity estimator, per-pixel PCG",
                   "image": [256, 256], "spp": spp, "bounces": bounces,
                   "triangles": 1282},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                     "traffic": None,
                     "kernel": "k_extend (closest-hit traversal)",
                     "launch_ms": mean_ms, "algorithmic_bytes_per_launch": per_launch_bytes,
                     "rays_per_step": rays, "slab_tests_per_ray": box / max(rays, 1),
                     "tri_tests_per_ray": tri / max(rays, 1)},
        "extra": {"gpu_ms_per_step": tot_ms / args.steps,
                  "Mrays_per_s": rays * args.steps / wall / 1e6,
                  "step_ms": steps_ms},
    }
    if not args.no_cpu:
        cpu = host_cpu()
        res["cpu_baseline"] = cpu_baseline_config1(cpu["threads"])
        res["cpu_baseline"]["host"] = cpu
    img.free()
    s.close()
    dev.close()
    return res


def cpu_baseline_box(desc, threads, spp=4, bounces=6, repeats=3):
    """The oracle on the same scene and estimator (plain unbiased tracer,
    per-pixel PCG) over the same SAH hierarchy (the reference's greedy
    builder is O(n^2 log n) and its 32/128 overlap buffers overflow at this
    scale), 64x64 tiles from an atomic counter on `threads` workers: one
    warm-up frame at 1 spp, then the median of `repeats` full frames at
    `spp`; plus one thread on a band of 64 rows at `spp`.  Scene and
    hierarchy build time is reported separately."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    from _libs import (SPO_EST_UNBIASED, SPO_HIT_REFERENCE, SPO_RNG_PCG,
                       SPO_TX_LIBM, SpoConfig, oracle)
    from _scenes import load_oracle

    O = oracle()
    t0 = time.perf_counter()
    s, cam = load_oracle(desc, sah=True)
    build_s = time.perf_counter() - t0
    w, h = desc["camera"][0], desc["camera"][1]

    def cfg_for(n):
        return SpoConfig(rng=SPO_RNG_PCG, tx=SPO_TX_LIBM, hit=SPO_HIT_REFERENCE,
                         estimator=SPO_EST_UNBIASED, samplesPerPixel=n,
                         bounces=bounces, radianceClamp=0.0, jitterYFirst=1,
                         seed=0x5EED)

    px = np.zeros(w * h * 4, np.float32)
    O.spo_render_threaded(s, C.byref(cam), C.byref(cfg_for(1)), 64, 64, threads, px,
                          np.zeros(12, np.uint64))
    secs, rays = [], 0
    cfg = cfg_for(spp)
    for _ in range(repeats):
        met = np.zeros(12, np.uint64)
        secs.append(O.spo_render_threaded(s, C.byref(cam), C.byref(cfg), 64, 64, threads,
                                          px, met))
        rays = int(met[2])
    sec = float(np.median(secs))
    band = min(64, h)
    t0 = time.perf_counter()
    O.spo_path_trace_tile(s, C.byref(cam), C.byref(cfg), 0, 0, w, band, None, px,
                          np.zeros(12, np.uint64))
    sec1 = time.perf_counter() - t0
    O.spo_scene_destroy(s)
    return {"value": w * h * spp / sec / 1e6, "unit": "Msamples/s", "cores": threads,
            "kind": "port",
            "sample": f"{w}x{h} frames at {spp} spp, {bounces} bounces, plain unbiased "
                      f"tracer, libm transcendentals, same SAH BVH; median of {repeats} "
                      f"after a 1-spp warm-up ({sec:.2f} s per frame)",
            "Mrays_per_s": rays / sec / 1e6,
            "value_1thread": w * band * spp / sec1 / 1e6,
            "sample_1thread": f"rows 0-{band - 1} at {spp} spp on one thread "
                              f"({sec1:.2f} s)",
            "scene_build_s": build_s}


def bench_box(args, V, scenes, name):
    """config5 (or config4): the plain (unbiased) GPU tracer, `--spp` samples
    per pixel per step over the whole image (config5: 1, the headline
    configuration; config4: 2, so that one launch holds 524,288 paths and
    fills the persistent grid's 327,680 lanes)."""
    dev = V.Device(0)
    desc = scenes.config5() if name == "config5" else scenes.config4()
    w, h = desc["camera"][0], desc["camera"][1]
    bounces = 6
    t0 = time.perf_counter()
    s, cam = scenes.load_gpu(dev, desc)
    build_s = time.perf_counter() - t0
    tiles = V.ComputeTiles(w, h, 64, 64)
    img = dev.alloc(w * h * 16)
    tx = V.TX_FAST if args.fast else V.TX_DOUBLE
    spp = args.spp or (1 if name == "config5" else 2)

    est = V.EST_NEE if args.estimator == "nee" else V.EST_UNBIASED

    def ctx_for(step, collect=False):
        return V.make_context(cam, s, spp=spp, bounces=bounces, clamp=0.0,
                              estimator=est, rng=V.RNG_PCG, seed=0x5EED,
                              transcendentals=tx, sample_offset=step * spp,
                              collect=collect)

    for k in range(args.warmup):
        V.path_trace_tiles_device(ctx_for(k), tiles, img)
    dev.synchronize()
    ext_ms, ext_n, sh_ms, tot_ms = 0.0, 0, 0.0, 0.0
    pcls = {"raygen": 0.0, "finalize": 0.0}
    t0 = time.perf_counter()
    for k in range(args.steps):
        V.path_trace_tiles_device(ctx_for(args.warmup + k), tiles, img)
        tim = dev.last_timings()
        ext_ms += tim["extend"][0]
        ext_n += tim["extend"][1]
        sh_ms += tim["shade"][0]
        tot_ms += tim["total"][0]
        for key in pcls:
            pcls[key] += tim[key][0]
    dev.synchronize()
    wall = time.perf_counter() - t0
    m = V.path_trace_tiles_device(ctx_for(args.warmup, collect=True), tiles, img)
    c = dev.last_counters()
    rays, box, tri = c["rays"], c["slab_tests"], c["tri_tests"]
    tbox, ment = c["tlas_slab_tests"], c["mesh_tests"]
    bytes_step = ((RAY_BYTES + HIT_BYTES_SCENE) * rays + BOX_BYTES * (box + tbox) +
                  TRI_BYTES * tri + ENTRY_BYTES * ment)
    # compulsory bytes of one launch: its rays in and hit records out, and
    # every mesh record (wide nodes and triangles, 64 bytes each) and
    # instance record (128 bytes) read once
    scene_bytes = sum(64 * sum(s.wide_counts(k)) for k in range(len(desc["meshes"])))
    scene_bytes += 128 * len(desc["objects"])
    launches = ext_n / args.steps
    per_launch = bytes_step / launches
    mean_ms = ext_ms / ext_n
    achieved = per_launch / (mean_ms * 1e-3) / 1e9
    counted = name == "config5" and est == V.EST_UNBIASED   # the counter runs' launches
    samples = w * h * spp
    res = {
        "metric": METRIC,
        "value": samples * args.steps / wall / 1e6,
        "unit": "Msamples/s",
        "ms_per_step": wall * 1e3 / args.steps,
        "dtype": "f32",
        "config": {"workload": f"{name}: {desc['triangles']} triangles ("
                               f"{len(desc['objects']) - 1} displaced icospheres of "
                               f"20480 in a closed box with a 1x1 opening), sky cube "
                               f"6x64x64 (sun 50), {w}x{h}, {spp} spp per step, "
                               f"{bounces} bounces, "
                               f"{'NEE' if args.estimator == 'nee' else 'plain unbiased'} "
                               f"tracer, per-pixel "
                               f"PCG, {'fast' if args.fast else 'double-evaluated'} "
                               f"transcendentals",
                   "image": [w, h], "spp_per_step": spp, "bounces": bounces,
                   "triangles": desc["triangles"]},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                     "traffic": (TRAFFIC_BYTES_PER_RAY["config5"] * rays / launches
                                 if counted else None),
                     "traffic_source": TRAFFIC_SOURCE if counted else None,
                     "traffic_frac": (TRAFFIC_BYTES_PER_RAY["config5"] * rays / launches /
                                      (mean_ms * 1e-3) / 1e9 / HBM_PEAK_GBS
                                      if counted else None),
                     "kernel": "k_extend (closest-hit traversal)",
                     "launch_ms": mean_ms, "algorithmic_bytes_per_launch": per_launch,
                     "compulsory_bytes_per_launch": (RAY_BYTES + HIT_BYTES_SCENE) * rays /
                     launches + scene_bytes,
                     "limiter": LIMITER.get(name) if counted else None,
                     "rays_per_step": rays, "slab_tests_per_ray": box / max(rays, 1),
                     "tri_tests_per_ray": tri / max(rays, 1),
                     "tlas_slab_tests_per_ray": tbox / max(rays, 1),
                     "mesh_entries_per_ray": ment / max(rays, 1)},
        "extra": {"Mrays_per_s": rays * args.steps / wall / 1e6,
                  "extend_ms_per_step": ext_ms / args.steps,
                  "shade_ms_per_step": sh_ms / args.steps,
                  "raygen_ms_per_step": pcls["raygen"] / args.steps,
                  "finalize_ms_per_step": pcls["finalize"] / args.steps,
                  "gpu_ms_per_step": tot_ms / args.steps,
                  "scene_build_s": build_s,
                  "paths_per_step": m.values[V.METRIC_PATHS]},
    }
    if args.no_guided:
        img.free()
        s.close()
        dev.close()
        return res
    # the guided tracer on the same workload: guide inference every bounce
    # and online training (stepsPerPass Adam steps) after every step; device
    # float transcendentals, as the time-to-relMSE runs use, with the plain
    # tracer in the same mode beside it
    gtx = V.TX_FAST
    g = V.Guide(dev, seed=1, max_weight=10.0)

    def gctx(step, train=True):
        return V.make_context(cam, s, spp=1, bounces=bounces, clamp=0.0,
                              estimator=V.EST_GUIDED, rng=V.RNG_PCG, seed=0x6EED,
                              transcendentals=gtx, sample_offset=step, guide=g,
                              train=train)

    pf_ms = 0.0
    for k in range(args.warmup + args.steps):
        V.path_trace_tiles_device(V.make_context(cam, s, spp=1, bounces=bounces,
                                                 clamp=0.0, estimator=V.EST_UNBIASED,
                                                 rng=V.RNG_PCG, seed=0x5EED,
                                                 transcendentals=gtx, sample_offset=k),
                                  tiles, img)
        if k >= args.warmup:
            pf_ms += dev.last_timings()["total"][0]

    for k in range(args.warmup):
        V.path_trace_tiles_device(gctx(k), tiles, img)
    dev.synchronize()
    cls = {"extend": 0.0, "shade": 0.0, "guide": 0.0, "total": 0.0}
    t0 = time.perf_counter()
    for k in range(args.steps):
        V.path_trace_tiles_device(gctx(args.warmup + k), tiles, img)
        tim = dev.last_timings()
        for key in cls:
            cls[key] += tim[key][0]
    dev.synchronize()
    gwall = time.perf_counter() - t0
    train_samples = g.samples()
    # inference only (frozen guide)
    fcls = {"raygen": 0.0, "extend": 0.0, "shade": 0.0, "finalize": 0.0, "guide": 0.0,
            "total": 0.0}
    infer_launches, evals = 0, 0
    t0 = time.perf_counter()
    for k in range(args.steps):
        V.path_trace_tiles_device(gctx(args.warmup + k, train=False), tiles, img)
        tim = dev.last_timings()
        for key in fcls:
            fcls[key] += tim[key][0]
        infer_launches += tim["guide"][1]
        evals += dev.last_counters()["guide_evals"]
    dev.synchronize()
    fwall = time.perf_counter() - t0
    # MFMA rooflines of the network: inference (k_guide_infer: 2 (64*64*4 +
    # 64*48) FLOP per evaluated hit, mean launch time from the trace's own
    # stamps) and one training step on this workload's collected samples
    # (k_guide_wsum + k_guide_fwdbwd + k_guide_wgrad +
    # k_guide_adam: about 3x the forward FLOP per sample; host wall clock
    # of 50 steps including launch gaps)
    flop_inf = 2 * (64 * 64 * 4 + 64 * 48)
    infer_ms = fcls["guide"] / max(infer_launches, 1)
    infer_flop = flop_inf * evals / max(infer_launches, 1)
    gt = V.Guide(dev, seed=1, max_weight=10.0)
    gt.train(train_samples, steps=5)
    dev.synchronize()
    t0 = time.perf_counter()
    gt.train(train_samples, steps=50)
    dev.synchronize()
    step_s = (time.perf_counter() - t0) / 50
    gt.close()
    train_flop = 3 * flop_inf * 16384
    res["extra"]["guide_mfma"] = {
        "peak_tflops": MFMA_FP16_PEAK_TFLOPS,
        "infer": {"kernel": "k_guide_infer", "launch_ms": infer_ms,
                  "evals_per_launch": evals / max(infer_launches, 1),
                  "flop_per_launch": infer_flop,
                  "achieved_tflops": infer_flop / (infer_ms * 1e-3) / 1e12,
                  "frac": infer_flop / (infer_ms * 1e-3) / 1e12 / MFMA_FP16_PEAK_TFLOPS},
        "train_step": {"kernels": "k_guide_wsum, k_guide_fwdbwd, k_guide_wgrad, "
                                  "k_guide_adam",
                       "batch": 16384, "step_ms": step_s * 1e3,
                       "flop_per_step": train_flop,
                       "achieved_tflops": train_flop / step_s / 1e12,
                       "frac": train_flop / step_s / 1e12 / MFMA_FP16_PEAK_TFLOPS,
                       "samples_from": f"{len(train_samples)} samples collected by the "
                                       f"last training pass of this workload"}}
    res["extra"]["guided"] = {
        "transcendentals": "device float",
        "plain_gpu_ms_per_step_same_mode": pf_ms / args.steps,
        "Msamples_per_s_training": samples * args.steps / gwall / 1e6,
        "Msamples_per_s_frozen": samples * args.steps / fwall / 1e6,
        "ms_per_step_training": gwall * 1e3 / args.steps,
        "ms_per_step_frozen": fwall * 1e3 / args.steps,
        "kernel_ms_per_step": {k: v / args.steps for k, v in cls.items()},
        "frozen_kernel_ms_per_step": {k: v / args.steps for k, v in fcls.items()},
        "training_steps_per_pass": 4, "batch": 16384,
        "collected_last_pass": g.stats()["collected"]}
    g.close()
    if name == "config5":
        # the full guided + batched form: the whole image as one batch item,
        # guide inference, sample collection and training captured in the
        # HIP graph; a step is one replay (one sample per pixel, one pass of
        # online training)
        gb = V.Guide(dev, seed=1, max_weight=10.0)
        b = V.Batch(dev, [(cam, s, img)], spp=1, bounces=bounces, clamp=0.0,
                    estimator=V.EST_GUIDED, rng=V.RNG_PCG, seed=0x6EED,
                    transcendentals=gtx, autotune=True, guide=gb, train=True)
        for _ in range(args.warmup):
            b.run()
        bms = 0.0
        t0 = time.perf_counter()
        for _ in range(args.steps):
            b.run()
            bms += b.last_ms()
        bwall = time.perf_counter() - t0
        res["extra"]["guided_batched"] = {
            "Msamples_per_s": samples * args.steps / bwall / 1e6,
            "ms_per_step": bwall * 1e3 / args.steps,
            "gpu_ms_per_step": bms / args.steps,
            "tuning": b.tuning(), "adam_steps": gb.stats()["steps"],
            "workload": "config5 image as one batch item, guided estimator with "
                        "online training, graph replays of one pass"}
        b.close()
        gb.close()
    if not args.no_cpu:
        cpu = host_cpu()
        res["cpu_baseline"] = cpu_baseline_box(desc, cpu["threads"], bounces=bounces)
        res["cpu_baseline"]["host"] = cpu
    img.free()
    s.close()
    dev.close()
    return res


def cpu_baseline_config3(descs, threads, budget_s=12.0):
    """The oracle (same estimator, SAH hierarchy) on the batch's scenes in
    order, 1 spp each, until about budget_s of rendering."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    from _libs import (SPO_EST_UNBIASED, SPO_HIT_REFERENCE, SPO_RNG_PCG,
                       SPO_TX_LIBM, SpoConfig, oracle)
    from _scenes import load_oracle

    O = oracle()
    cfg = SpoConfig(rng=SPO_RNG_PCG, tx=SPO_TX_LIBM, hit=SPO_HIT_REFERENCE,
                    estimator=SPO_EST_UNBIASED, samplesPerPixel=1, bounces=5,
                    radianceClamp=0.0, jitterYFirst=1, seed=0x5EED)
    total_s, samples, used = 0.0, 0, 0
    for d in descs:
        s, cam = load_oracle(d, sah=True)
        w, h = d["camera"][0], d["camera"][1]
        px = np.zeros(w * h * 4, np.float32)
        total_s += O.spo_render_threaded(s, C.byref(cam), C.byref(cfg), 64, 64, threads,
                                         px, np.zeros(12, np.uint64))
        O.spo_scene_destroy(s)
        samples += w * h
        used += 1
        if total_s > budget_s:
            break
    return {"value": samples / total_s / 1e6, "unit": "Msamples/s", "cores": threads,
            "kind": "port",
            "sample": f"the first {used} scenes of the set at 1 spp, 5 bounces, plain "
                      f"unbiased tracer over the same SAH BVHs ({samples} samples, "
                      f"{total_s:.1f} s)"}


def bench_config3(args, V, scenes):
    """The batched workload: 64 scenes rendered as one wavefront from a
    captured HIP graph, 16 spp, 5 bounces; a step is one replay (every
    scene's image)."""
    dev = V.Device(0)
    descs = scenes.config3()
    t0 = time.perf_counter()
    loaded = [scenes.load_gpu(dev, d) for d in descs]
    build_s = time.perf_counter() - t0
    imgs = [dev.alloc(d["camera"][0] * d["camera"][1] * 16) for d in descs]
    items = [(cam, s, img) for (s, cam), img in zip(loaded, imgs)]
    spp, bounces = 16, 5
    t0 = time.perf_counter()
    b = V.Batch(dev, items, spp=spp, bounces=bounces, clamp=0.0,
                estimator=V.EST_UNBIASED, rng=V.RNG_PCG, seed=0x5EED,
                transcendentals=V.TX_FAST, autotune=True)
    create_s = time.perf_counter() - t0
    tuning = b.tuning()
    for _ in range(args.warmup):
        b.run()
    gpu_ms = 0.0
    t0 = time.perf_counter()
    for _ in range(args.steps):
        m = b.run()
        gpu_ms += b.last_ms()
    wall = time.perf_counter() - t0
    pixels = tuning["pixels"]
    samples = pixels * spp
    # per-kernel times of the same render (eager) and its test counts
    tim, _ = b.profile(collect=False)
    _, cnt = b.profile(collect=True)
    rays = cnt["rays"]
    bytes_render = ((RAY_BYTES + HIT_BYTES_SCENE) * rays +
                    BOX_BYTES * (cnt["slab_tests"] + cnt["tlas_slab_tests"]) +
                    TRI_BYTES * cnt["tri_tests"] + ENTRY_BYTES * cnt["mesh_tests"])
    ext_ms, ext_n = tim["extend"]
    per_launch = bytes_render / ext_n
    mean_ms = ext_ms / ext_n
    achieved = per_launch / (mean_ms * 1e-3) / 1e9
    tris = [d["triangles"] for d in descs]
    sides = [d["camera"][0] for d in descs]
    res = {
        "metric": METRIC,
        "value": samples * args.steps / wall / 1e6,
        "unit": "Msamples/s",
        "ms_per_step": wall * 1e3 / args.steps,
        "dtype": "f32",
        "config": {"workload": f"config3: {len(descs)} seeded scenes of noise-displaced "
                               f"icospheres on jittered instance grids over a ground "
                               f"quad ({min(tris)}..{max(tris)} triangles), square "
                               f"images {min(sides)}..{max(sides)} px ({pixels} pixels "
                               f"in all), {spp} spp, {bounces} bounces, Lambert albedo "
                               f"U[0.1,0.9], sky cube with sun; one wavefront over all "
                               f"scenes replayed from a HIP graph, launch shape "
                               f"autotuned",
                   "scenes": len(descs), "pixels": pixels, "spp": spp,
                   "bounces": bounces, "tuning": tuning},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS, "traffic": None,
                     "kernel": "k_extend (closest-hit traversal, batch variant)",
                     "launch_ms": mean_ms, "launches_per_step": ext_n,
                     "algorithmic_bytes_per_launch": per_launch,
                     "rays_per_step": rays,
                     "slab_tests_per_ray": cnt["slab_tests"] / max(rays, 1),
                     "tlas_slab_tests_per_ray": cnt["tlas_slab_tests"] / max(rays, 1),
                     "tri_tests_per_ray": cnt["tri_tests"] / max(rays, 1),
                     "mesh_entries_per_ray": cnt["mesh_tests"] / max(rays, 1)},
        "extra": {"gpu_ms_per_step": gpu_ms / args.steps,
                  "Mrays_per_s": m.values[V.METRIC_RAYS] * args.steps / wall / 1e6,
                  "eager_kernel_ms": {k: v[0] for k, v in tim.items()},
                  "scene_build_s": build_s, "batch_create_s": create_s},
    }
    if not args.no_cpu:
        cpu = host_cpu()
        res["cpu_baseline"] = cpu_baseline_config3(descs, cpu["threads"])
        res["cpu_baseline"]["host"] = cpu
    b.close()
    for img in imgs:
        img.free()
    for s, _ in loaded:
        s.close()
    dev.close()
    return res


# ---------------------------------------------------------------- relMSE
def relmse(img, ref):
    """Relative MSE, mean over pixels and channels of (x - r)^2 / (r^2 +
    0.01) (the convention of the path-guiding literature, e.g. Mueller et
    al. 2017)."""
    return float(np.mean((img - ref) ** 2 / (ref * ref + 1e-2)))


class DeviceAccumulator:
    """Renders chunks of samples of one scene and keeps their running mean
    on the device (spg_accumulate_device).  `wall` is the host wall clock
    around the render and accumulate calls (each trace call returns when its
    work is done); reading the mean back for a relMSE checkpoint is outside
    it."""

    def __init__(self, V, dev, s, cam, w, h, bounces=6):
        self.V, self.dev, self.s, self.cam, self.w, self.h = V, dev, s, cam, w, h
        self.bounces = bounces
        self.tiles = V.ComputeTiles(w, h, 64, 64)
        self.img = dev.alloc(w * h * 16)
        self.acc = dev.upload(np.zeros(w * h * 4, np.float32))
        self.spp = 0
        self.wall = 0.0

    def add(self, spp, est, seed, guide=None, train=False):
        V = self.V
        t0 = time.perf_counter()
        ctx = V.make_context(self.cam, self.s, spp=spp, bounces=self.bounces, clamp=0.0,
                             estimator=est, rng=V.RNG_PCG, seed=seed,
                             sample_offset=self.spp, transcendentals=V.TX_FAST,
                             guide=guide, train=train)
        V.path_trace_tiles_device(ctx, self.tiles, self.img)
        self.dev.accumulate(self.acc, self.img, self.w * self.h, self.spp, spp)
        self.dev.synchronize()
        self.wall += time.perf_counter() - t0
        self.spp += spp

    def mean(self):
        px = self.acc.download(np.float32, self.w * self.h * 4)
        return px.reshape(self.h, self.w, 4)[:, :, :3].astype(np.float64)

    def close(self):
        self.img.free()
        self.acc.free()


def render_reference(V, dev, s, cam, w, h, spp, est, chunk=256):
    """The reference image: two independent halves of `spp` samples (the
    unbiased estimator `est`, different seeds), averaged.  Its own relMSE
    against the true image is estimated as relMSE(half A, half B) / 4 (the
    halves' difference has twice one half's variance; the average has half
    of it)."""
    halves, wall = [], 0.0
    for seed in (0xA11CE, 0xB0B):
        acc = DeviceAccumulator(V, dev, s, cam, w, h)
        while acc.spp < spp // 2:
            acc.add(min(chunk, spp // 2 - acc.spp), est, seed)
            if acc.spp % 4096 == 0:
                log(f"reference half {len(halves) + 1}: {acc.spp} spp, {acc.wall:.1f} s")
        halves.append(acc.mean())
        wall += acc.wall
        acc.close()
        log(f"reference half {len(halves)}: {spp // 2} spp in {acc.wall:.1f} s")
    floor = relmse(halves[0], halves[1]) / 4.0
    return (halves[0] + halves[1]) / 2.0, floor, wall


def crossing(curve, target):
    """Wall time and spp at which `relmse` (the reference's own error
    subtracted) reaches `target`: log-log interpolation between the two
    checkpoints around the crossing ("measured"), or beyond the last
    checkpoint with the error falling as 1/spp and time growing at the last
    segment's rate ("extrapolated")."""
    prev = None
    for c in curve:
        t, n, e = c["wall_s"], c["spp"], c["relmse_true"]
        if e <= target:
            if prev is None:
                return t, n, "measured"
            t0, n0, e0 = prev
            f = (np.log(target) - np.log(e0)) / (np.log(e) - np.log(e0))
            return (float(np.exp(np.log(t0) + f * (np.log(t) - np.log(t0)))),
                    float(np.exp(np.log(n0) + f * (np.log(n) - np.log(n0)))),
                    "measured")
        prev = (t, n, max(e, 1e-12))
    if len(curve) < 2:
        return None
    a, b = curve[-2], curve[-1]
    need = b["spp"] * b["relmse_true"] / target
    rate = (b["wall_s"] - a["wall_s"]) / (b["spp"] - a["spp"])
    return b["wall_s"] + (need - b["spp"]) * rate, need, "extrapolated"


def time_to_relmse(V, dev, scenes, workload, ref_spp, ref_est, max_spp=8192,
                   train_passes=64, guide_kw=None, target=1e-3):
    """Wall-clock time to relMSE `target` of the plain tracer, the guided
    tracer (online training during its first `train_passes` one-sample
    passes, then the frozen guide), next-event estimation (learning its
    sky / emitter split from its own calls) and the guided tracer with
    next-event estimation (trained the same way, the split learned by its
    training passes), each
    accumulating every sample it renders, against a reference of `ref_spp`
    samples of `ref_est` rendered here."""
    desc = getattr(scenes, workload)()
    w, h = desc["camera"][0], desc["camera"][1]
    s, cam = scenes.load_gpu(dev, desc)
    ref, floor, ref_wall = render_reference(V, dev, s, cam, w, h, ref_spp, ref_est)
    guide_kw = guide_kw or dict(seed=1, learning_rate=3e-3, batch_size=16384,
                                steps_per_pass=4, max_weight=10.0)

    def run(name, step):
        acc = DeviceAccumulator(V, dev, s, cam, w, h)
        curve, nxt = [], 16
        while acc.spp < max_spp:
            step(acc)
            if acc.spp >= nxt:
                e = relmse(acc.mean(), ref)
                curve.append({"wall_s": acc.wall, "spp": acc.spp, "relmse": e,
                              "relmse_true": max(e - floor, 0.0)})
                log(f"{workload} {name}: {acc.spp} spp, {acc.wall:.2f} s, relMSE {e:.5f}")
                nxt *= 2
                if e - floor < target / 2:
                    break
        acc.close()
        return curve

    plain = run("plain", lambda a: a.add(64 if a.spp >= 64 else 16, V.EST_UNBIASED,
                                         0x5EED))
    g = V.Guide(dev, **guide_kw)

    def guided_step(a):
        if a.spp < train_passes:
            a.add(1, V.EST_GUIDED, 0x6EED, guide=g, train=True)
        else:
            a.add(64, V.EST_GUIDED, 0x6EED, guide=g)

    guided = run("guided", guided_step)
    g.close()
    s.learn_light_split(True)  # NEE learns its sky / emitter split from its own calls
    nee = run("nee", lambda a: a.add(64 if a.spp >= 64 else 16, V.EST_NEE, 0x7EED))
    nee_split = s.light_split()
    s.learn_light_split(False)
    g = V.Guide(dev, **guide_kw)

    def guided_nee_step(a):
        if a.spp < train_passes:
            a.add(1, V.EST_GUIDED_NEE, 0x8EED, guide=g, train=True)
        else:
            a.add(64, V.EST_GUIDED_NEE, 0x8EED, guide=g)

    guided_nee = run("guided+nee", guided_nee_step)
    learned_split = g.light_split()
    g.close()
    s.close()
    res = {"workload": workload, "target": target, "wall_clock": True,
           "reference": {"spp": ref_spp,
                         "estimator": {V.EST_UNBIASED: "plain", V.EST_NEE: "nee"}[ref_est],
                         "own_relmse": floor, "render_s": ref_wall},
           "train_passes": train_passes, "guide": guide_kw}
    for name, curve in (("plain", plain), ("guided", guided), ("nee", nee),
                        ("guided_nee", guided_nee)):
        c = crossing(curve, target)
        res[name] = {"time_s": c[0] if c else None, "spp": c[1] if c else None,
                     "how": c[2] if c else None, "curve": curve}
    res["guided_nee"]["light_split"] = learned_split
    res["nee"]["light_split"] = nee_split
    tp = res["plain"]["time_s"]
    for name in ("guided", "nee", "guided_nee"):
        t = res[name]["time_s"]
        res[name]["speedup_vs_plain"] = tp / t if tp and t else None
    return res


def bench_relmse(args, V, scenes):
    """`--relmse`: the time-to-relMSE measurement alone on the workload."""
    dev = V.Device(0)
    ref_est = V.EST_NEE if args.ref_estimator == "nee" else V.EST_UNBIASED
    res = time_to_relmse(V, dev, scenes, args.workload, args.ref_spp, ref_est,
                         max_spp=args.max_spp, train_passes=args.train_passes,
                         guide_kw=dict(seed=args.guide_seed, learning_rate=args.guide_lr,
                                       batch_size=args.guide_batch,
                                       steps_per_pass=args.guide_steps,
                                       max_weight=args.guide_max_weight,
                                       bsdf_fraction=args.guide_bsdf))
    print(json.dumps(res))
    dev.close()


def bench_soup(args, V, scenes):
    dev = V.Device(0)
    tris, o, d = scenes.soup(1_000_000, 1 << 22, seed=7)
    s = V.Scene(dev)
    v, i = scenes.soup_mesh(tris)
    m = s.create_mesh(v, i, smooth=False)
    s.build()
    n = len(o)
    bufs = [dev.upload(np.ascontiguousarray(x)) for x in
            (o[:, 0], o[:, 1], o[:, 2], d[:, 0], d[:, 1], d[:, 2])]
    outp, outt = dev.alloc(4 * n), dev.alloc(4 * n)
    st = V.TraversalStats()
    V.check(V.lib().spg_intersect_closest_device(
        s.handle, m, *[b.ptr for b in bufs], n, outp.ptr, outt.ptr, None, None,
        C.byref(st)))
    ms = C.c_double()
    for _ in range(args.warmup):
        V.check(V.lib().spg_intersect_closest_device(
            s.handle, m, *[b.ptr for b in bufs], n, outp.ptr, outt.ptr, None, None, None))
    t0 = time.perf_counter()
    V.check(V.lib().spg_time_intersect_closest(s.handle, m, *[b.ptr for b in bufs], n,
                                               outp.ptr, outt.ptr, args.steps,
                                               C.byref(ms)))
    wall = time.perf_counter() - t0
    bytes_launch = ((RAY_BYTES + HIT_BYTES_MESH) * n + BOX_BYTES * st.boxTests +
                    TRI_BYTES * st.triTests)
    achieved = bytes_launch / (ms.value * 1e-3) / 1e9
    res = {
        "metric": "Mrays/s (closest hit)",
        "value": n * args.steps / wall / 1e6,
        "unit": "Mrays/s",
        "ms_per_step": wall * 1e3 / args.steps,
        "dtype": "f32",
        "config": {"workload": "soup: 2^22 rays (origins U[-2,2]^3, directions "
                               "uniform on S^2) vs 1M triangles (centroids U[0,1]^3, "
                               "edge lognormal(-5, 0.5)), SAH BVH2"},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                     "traffic": TRAFFIC_BYTES_PER_RAY["soup"] * n,
                     "traffic_source": TRAFFIC_SOURCE, "kernel": "k_closest_mesh",
                     "launch_ms": ms.value, "algorithmic_bytes_per_launch": bytes_launch,
                     "slab_tests_per_ray": st.boxTests / n,
                     "tri_tests_per_ray": st.triTests / n},
    }
    if not args.no_cpu:
        cpu = host_cpu()
        res["cpu_baseline"] = cpu_baseline_soup(cpu["threads"], tris, o, d)
        res["cpu_baseline"]["host"] = cpu
    for b in bufs + [outp, outt]:
        b.free()
    s.close()
    dev.close()
    return res


def bench_irradiance(args, V, scenes):
    """CreateIrradianceCubeMap on the reference's call (src/main.cpp:1313:
    32x32 faces) from a 2048x1024 synthetic HDR sky (sky gradient + sun of
    radiance 50, above the radiance clamp of 10): one step = the whole cube
    map; double-evaluated transcendentals (the oracle-exact mode)."""
    dev = V.Device(0)
    ew, eh, fw, fh = 2048, 1024, 32, 32
    sky = V.gen_sky_equirect(ew, eh).reshape(eh, ew, 4)
    tx = V.TX_FAST if args.fast else V.TX_DOUBLE
    for _ in range(max(1, args.warmup)):
        dev.create_irradiance_cubemap(sky, fw, fh, 10.0, tx)
    kms = []
    t0 = time.perf_counter()
    for _ in range(args.steps):
        _, ms = dev.create_irradiance_cubemap(sky, fw, fh, 10.0, tx)
        kms.append(ms)
    wall = time.perf_counter() - t0
    samples = 6 * fw * fh * 63 * 16
    kernel_ms = float(np.mean(kms))
    # algorithmic bytes: the four RGBA32F texels of every bilinear lookup
    # and the output texel (what an implementation without caches would move)
    bytes_launch = samples * 64 + 6 * fw * fh * 16
    achieved = bytes_launch / (kernel_ms * 1e-3) / 1e9
    res = {
        "metric": "Gsamples/s (irradiance cube map, kernel)",
        "value": samples / (kernel_ms * 1e-3) / 1e9,
        "unit": "Gsamples/s",
        "ms_per_step": wall * 1e3 / args.steps,
        "dtype": "f32 (f64 transcendentals)" if tx == V.TX_DOUBLE else "f32",
        "config": {"workload": f"irradiance cube map: 6 faces of {fw}x{fh} from a "
                               f"{ew}x{eh} RGBA32F sky equirect, 63x16 samples per "
                               "texel, radiance clamp 10",
                   "samples_per_step": samples},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS, "traffic": None,
                     "kernel": "k_irradiance", "launch_ms": kernel_ms,
                     "algorithmic_bytes_per_launch": bytes_launch},
        "extra": {"step_ms_with_copies": wall * 1e3 / args.steps},
    }
    if not args.no_cpu:
        res["cpu_baseline"] = cpu_baseline_irradiance(sky, fw, fh)
    dev.close()
    return res


def bench_copy(args, V, scenes):
    """Calibration workload for HBM counters: a plain device-to-device copy
    of 1 GiB (torch's elementwise copy kernel on cuda:0), `steps` times.  A
    rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE pass over this command gives what
    the counters read for 1 GiB read and 1 GiB written, the factors that
    scale the same counters of the tracer's kernels into bytes."""
    import torch

    n = 1 << 28  # floats: 1 GiB
    src = torch.rand(n, device="cuda:0")
    dst = torch.empty_like(src)
    for _ in range(max(1, args.warmup)):
        dst.copy_(src)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        dst.copy_(src)
    torch.cuda.synchronize()
    sec = (time.perf_counter() - t0) / args.steps
    ok = bool(torch.equal(dst, src))
    return {"metric": "GB/s (1 GiB device copy, read + write)",
            "value": 2 * 4 * n / sec / 1e9, "unit": "GB/s", "ms_per_step": sec * 1e3,
            "dtype": "f32", "config": {"workload": "copy: 1 GiB device to device, "
                                                   "torch elementwise copy kernel",
                                       "bytes_read": 4 * n, "bytes_written": 4 * n,
                                       "equal": ok}}


def bench_tiles(args, V, scenes):
    """The drop-in path as the reference's worker pool drives it
    (src/main.cpp:731-759, src/config.h:21): 16 host threads pull 64x64
    tiles of the config5 image from a shared counter and call
    spg_path_trace_tile on one shared context, each tile's pixels written
    into one host image (host memory: the rate includes the device-to-host
    copies).  One step = every tile once at 1 spp, 6 bounces, plain
    unbiased tracer, double-evaluated transcendentals (the headline
    configuration).  Also: the same frame as one spg_path_trace_tiles call
    into host memory, and the device-resident call of the headline line."""
    import threading

    dev = V.Device(0)
    desc = scenes.config5()
    w, h = desc["camera"][0], desc["camera"][1]
    s, cam = scenes.load_gpu(dev, desc)
    tiles = V.ComputeTiles(w, h, 64, 64)
    img = np.zeros(w * h * 4, np.float32)
    threads = 16

    def ctx_for(step):
        return V.make_context(cam, s, spp=1, bounces=6, clamp=0.0,
                              estimator=V.EST_UNBIASED, rng=V.RNG_PCG, seed=0x5EED,
                              transcendentals=V.TX_DOUBLE, sample_offset=step)

    def pool_frame(ctx):
        lock = threading.Lock()
        nxt = [0]
        errors = []

        def work():
            try:
                while True:
                    with lock:
                        i = nxt[0]
                        nxt[0] += 1
                    if i >= len(tiles):
                        return
                    V.sp_PathTraceTile(ctx, tiles[i], img)
            except Exception as e:  # noqa: BLE001 - raised below
                errors.append(e)

        ts = [threading.Thread(target=work) for _ in range(threads)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        if errors:
            raise errors[0]

    for k in range(args.warmup):
        pool_frame(ctx_for(k))
    t0 = time.perf_counter()
    for k in range(args.steps):
        pool_frame(ctx_for(args.warmup + k))
    wall = time.perf_counter() - t0
    # the same frames as one batched host-memory call each, and device-resident
    t1 = time.perf_counter()
    for k in range(args.steps):
        V.path_trace_tiles(ctx_for(args.warmup + k), tiles, img)
    wall_batched = time.perf_counter() - t1
    dimg = dev.alloc(w * h * 16)
    V.path_trace_tiles_device(ctx_for(0), tiles, dimg)
    dev.synchronize()
    t2 = time.perf_counter()
    for k in range(args.steps):
        V.path_trace_tiles_device(ctx_for(args.warmup + k), tiles, dimg)
    dev.synchronize()
    wall_device = time.perf_counter() - t2
    dimg.free()
    samples = w * h
    res = {
        "metric": "Msamples/s through the drop-in tile call (16 host threads, "
                  "64x64 tiles, host image)",
        "value": samples * args.steps / wall / 1e6,
        "unit": "Msamples/s",
        "ms_per_step": wall * 1e3 / args.steps,
        "dtype": "f32",
        "config": {"workload": f"config5: {desc['triangles']} triangles, {w}x{h}, "
                               f"{len(tiles)} tiles of 64x64 traced by {threads} "
                               f"host threads calling spg_path_trace_tile on one "
                               f"shared context into host memory, 1 spp per "
                               f"frame, 6 bounces, plain unbiased tracer, "
                               f"double-evaluated transcendentals",
                   "tiles": len(tiles), "threads": threads},
        "extra": {"tiles_per_s": len(tiles) * args.steps / wall,
                  "batched_host_call_Msamples_per_s":
                      samples * args.steps / wall_batched / 1e6,
                  "device_resident_Msamples_per_s":
                      samples * args.steps / wall_device / 1e6,
                  "image_bytes_to_host_per_frame": 16 * samples},
    }
    s.close()
    dev.close()
    return res


def bench_post(args, V, scenes):
    """The step after the path on a 1920x1080 RGBA32F image: progressive
    accumulation of a new image into the running mean, then the viewer's
    tone mapping to RGBA8 (one step = both), plus the OBJ parser's host
    throughput on an 81,920-triangle mesh written as text."""
    dev = V.Device(0)
    w, h = 1920, 1080
    n = w * h
    rng = np.random.default_rng(1)
    a = rng.exponential(1.0, n * 4).astype(np.float32)
    b = rng.exponential(1.0, n * 4).astype(np.float32)
    acc, new = dev.upload(a), dev.upload(b)
    out = dev.alloc(4 * n)
    tx = V.TX_FAST if args.fast else V.TX_DOUBLE
    for _ in range(max(1, args.warmup)):
        dev.accumulate(acc, new, n, 1, 1)
        V.check(V.lib().spg_tonemap_device(dev.handle, acc.ptr, n, 1.0, tx, out.ptr))
    t0 = time.perf_counter()
    for k in range(args.steps):
        dev.accumulate(acc, new, n, k + 1, 1)
        V.check(V.lib().spg_tonemap_device(dev.handle, acc.ptr, n, 1.0, tx, out.ptr))
    wall = (time.perf_counter() - t0) / args.steps
    # kernel times from HIP events on the library's stream
    ka, kt = C.c_double(), C.c_double()
    V.check(V.lib().spg_time_post(dev.handle, acc.ptr, new.ptr, n, 1.0, tx, out.ptr,
                                  args.steps, C.byref(ka), C.byref(kt)))
    t_acc, t_tm = ka.value * 1e-3, kt.value * 1e-3
    # algorithmic bytes: accumulate reads two RGBA32F texels and writes one
    # (48 B/pixel); tone mapping reads one and writes an RGBA8 texel (20 B)
    bytes_acc, bytes_tm = n * 48, n * 20
    # OBJ text of a displaced level-6 icosphere
    v, idx = scenes.displaced_icosphere(6, seed=2)[:2]
    v = np.asarray(v, np.float32).reshape(-1, 8)
    lines = ["o mesh"] + ["v %.9g %.9g %.9g" % tuple(p[:3]) for p in v] + \
        ["vn %.9g %.9g %.9g" % tuple(p[3:6]) for p in v] + \
        ["f %d//%d %d//%d %d//%d" % (i + 1, i + 1, j + 1, j + 1, k + 1, k + 1)
         for i, j, k in np.asarray(idx).reshape(-1, 3)]
    text = ("\n".join(lines) + "\n").encode()
    t0 = time.perf_counter()
    _, pi = V.parse_obj(text)
    t_obj = time.perf_counter() - t0
    achieved = bytes_tm / t_tm / 1e9
    res = {
        "metric": "Mpixels/s (accumulate + tone map, 1080p)",
        "value": n / (t_acc + t_tm) / 1e6,
        "unit": "Mpixels/s",
        "ms_per_step": (t_acc + t_tm) * 1e3,
        "dtype": "f32 -> u8 (bytes of the f64 pow)" if tx == V.TX_DOUBLE else "f32 -> u8",
        "config": {"workload": "post step on 1920x1080 RGBA32F: running mean of two "
                               "images, then Reinhard + gamma 1/2.2 to RGBA8"},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS,
                     "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS, "traffic": None,
                     "kernel": "k_tonemap", "launch_ms": t_tm * 1e3,
                     "algorithmic_bytes_per_launch": bytes_tm},
        "extra": {"accumulate_ms": t_acc * 1e3, "tonemap_ms": t_tm * 1e3,
                  "accumulate_GBs": bytes_acc / t_acc / 1e9,
                  "step_ms_with_host_sync": wall * 1e3,
                  "obj_parse": {"triangles": int(len(pi) // 3), "bytes": len(text),
                                "ms": t_obj * 1e3,
                                "Mtris_per_s": len(pi) / 3 / t_obj / 1e6}},
    }
    if not args.no_cpu:
        sys.path.insert(0, os.path.join(ROOT, "tests"))
        from _libs import oracle
        O = oracle()
        d, q = a.copy(), np.zeros(n * 4, np.uint8)
        t0 = time.perf_counter()
        O.spo_accumulate(d, b, n, 1, 1)
        O.spo_tonemap(d, n, 1.0, 1 if tx == V.TX_DOUBLE else 0, q)
        sec = time.perf_counter() - t0
        res["cpu_baseline"] = {"value": n / sec / 1e6, "unit": "Mpixels/s", "cores": 1,
                               "kind": "port", "sample": f"one 1080p step ({sec:.2f} s)"}
    for buf in (acc, new, out):
        buf.free()
    dev.close()
    return res


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", default="config5",
                    choices=["config5", "config4", "config3", "config1", "soup",
                             "irradiance", "post", "copy", "tiles"])
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--fast", action="store_true",
                    help="device float transcendentals instead of double-evaluated")
    ap.add_argument("--relmse", action="store_true",
                    help="measure wall-clock time to relMSE 1e-3 of the plain, "
                         "guided and NEE tracers on the workload (config4 or "
                         "config5) instead, against a reference rendered in "
                         "the same run")
    ap.add_argument("--spp", type=int, default=None,
                    help="config4/config5: samples per pixel per step of the plain "
                         "tracer (default 1 on config5, 2 on config4)")
    ap.add_argument("--estimator", choices=["unbiased", "nee"], default="unbiased",
                    help="config4/config5: the first tracer's estimator")
    ap.add_argument("--no-guided", action="store_true",
                    help="config4/config5: the plain tracer only (for counter runs)")
    ap.add_argument("--no-relmse", action="store_true",
                    help="skip the config-4 time-to-relMSE part of the default run")
    ap.add_argument("--ref-spp", type=int, default=None,
                    help="reference samples per pixel (config4: 4096 NEE, "
                         "config5: 32768 plain)")
    ap.add_argument("--ref-estimator", choices=["plain", "nee"], default=None)
    ap.add_argument("--max-spp", type=int, default=8192)
    ap.add_argument("--train-passes", type=int, default=None,
                    help="one-sample passes of online training before the guide "
                         "is frozen (default 64 on config4, 256 on config5)")
    ap.add_argument("--guide-lr", type=float, default=None,
                    help="Adam learning rate (default 3e-3 on config4, 1e-2 on "
                         "config5)")
    ap.add_argument("--guide-batch", type=int, default=None,
                    help="training samples per Adam step (default 16384 on "
                         "config4, 65536 on config5)")
    ap.add_argument("--guide-steps", type=int, default=4)
    ap.add_argument("--guide-max-weight", type=float, default=10.0)
    ap.add_argument("--guide-seed", type=int, default=1)
    ap.add_argument("--guide-bsdf", type=float, default=0.5,
                    help="probability of the BSDF sampler in the guided "
                         "estimator's one-sample MIS")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported "
              "(this build traces on a single MI355X)", file=sys.stderr)
        sys.exit(2)
    import vk_cinematic_amd as V
    from vk_cinematic_amd import scenes

    if args.relmse:
        if args.workload not in ("config4", "config5"):
            sys.exit("--relmse measures config4 or config5")
        if args.ref_spp is None:
            args.ref_spp = 4096 if args.workload == "config4" else 32768
        if args.ref_estimator is None:
            args.ref_estimator = "nee" if args.workload == "config4" else "plain"
        if args.train_passes is None:
            args.train_passes = 64 if args.workload == "config4" else 256
        # config 5 trains longer on more samples per step (a sweep of
        # learning rate, batch and steps per pass on it: 1e-2 and 65,536
        # reach relMSE 1e-3 with 9% fewer samples than 3e-3 and 16,384)
        if args.guide_lr is None:
            args.guide_lr = 3e-3 if args.workload == "config4" else 1e-2
        if args.guide_batch is None:
            args.guide_batch = 16384 if args.workload == "config4" else 65536
        return bench_relmse(args, V, scenes)
    if args.workload in ("config5", "config4"):
        res = bench_box(args, V, scenes, args.workload)
    else:
        res = {"config1": bench_config1, "config3": bench_config3,
               "soup": bench_soup, "irradiance": bench_irradiance,
               "post": bench_post, "copy": bench_copy,
               "tiles": bench_tiles}[args.workload](
                   args, V, scenes)
    if args.workload == "config5" and not args.no_relmse:
        # the second half of the metric: wall-clock time to relMSE 1e-3,
        # guided vs plain, on the config-4 workload (the config-5 figure:
        # python bench.py --workload config5 --relmse)
        dev = V.Device(0)
        res["time_to_relmse"] = time_to_relmse(V, dev, scenes, "config4", 4096,
                                               V.EST_NEE, max_spp=4096)
        dev.close()
    out = {"metric": res.pop("metric"), "value": res.pop("value"),
           "unit": res.pop("unit"), "n_gpus": 1, "steps": args.steps,
           "warmup": args.warmup, "ms_per_step": res.pop("ms_per_step"),
           "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
           "dtype": res.pop("dtype"), "data": "synthetic"}
    out.update(res)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
