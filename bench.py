"""Closest-hit throughput on the diced-patch heightfield scene.

Workload (one step): one closest-hit trace of a 2^22-ray stream against the
64x64 bilinear-patch heightfield (psychopath_cpp_amd.configs.heightfield_scene,
split-diced at dice_rate 1.0): 2^21 primary rays (1024x1024, 2 samples per
pixel, Halton sample streams) followed by 2^21 cosine-distributed Lambert
first-bounce rays from their hits (sample dimensions 9 and 10).  The stream
is generated on the GPU and is resident in HBM before timing starts; it is
traced in its 56-byte-per-ray form (origin, direction, max_t, time, six
footprint terms) and writes 16 bytes per ray (t, instance, u, v).

Prints one JSON line.  `roofline` prices the trace's main pass, the
dominant kernel, against HBM (72 algorithmic bytes per ray, 8 TB/s), with
its duration from HIP events that the library records on the stream it
launches on; `traffic` is that kernel's measured HBM bytes per launch from
the committed rocprofv3 counter summary.  `cpu_baseline` times the oracle's
restatement of the reference's breadth-first CPU tracer on a sample of the
same stream, on this host's cores.
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

BYTES_PER_RAY = 72          # 56 B ray in + 16 B hit out
HBM_PEAK_GBS = 8000.0       # MI355X HBM3E
STREAM_RAYS = 1 << 22
W, H, SPP, SEED = 1024, 1024, 2, 1
METRIC = "closest-hit Mrays/s + %HBM roofline on diced-patch scene"


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def make_stream(ctx, scene):
    import torch
    from psychopath_cpp_amd import gpu
    prim, _ = gpu.camera_rays(ctx, scene, W, H, SPP, SEED)
    hits = gpu.trace_world(ctx, scene, prim)
    bounce, valid = gpu.bounce_rays(ctx, scene, prim, hits, W, SPP, SEED, 9, 10)
    idx = torch.nonzero(valid, as_tuple=False).flatten()
    nb = STREAM_RAYS - prim.shape[1]
    if idx.numel() == 0:
        raise RuntimeError("no valid bounce rays")
    # every primary ray of this camera lands on the field; if some bounce is
    # invalid, the valid ones are repeated cyclically to keep 2^21 rays
    idx = idx.repeat((nb + idx.numel() - 1) // idx.numel())[:nb]
    wrays = torch.cat([prim, bounce[:, idx]], dim=1).contiguous()
    return wrays, int(valid.sum().item())


def host_threads():
    """Host cores this process may use: its CPU affinity (what `nproc`
    reports), capped by OMP_NUM_THREADS where the host sets it (a shared
    GPU host sets it to the CPU share of one GPU)."""
    n = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    omp = os.environ.get("OMP_NUM_THREADS", "")
    if omp.isdigit() and int(omp) > 0:
        n = min(n, int(omp))
    return max(1, n)


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def mixed_sample(n_total, sample):
    """Indices of an equal mix of the stream's two halves: the first
    sample/2 primary rays and the first sample/2 bounce rays."""
    import numpy as np
    half = sample // 2
    return np.concatenate([np.arange(half), n_total // 2 + np.arange(sample - half)])


def cpu_baseline(scene_py, wrays, pick, min_seconds):
    """The oracle's breadth-first tracer on the rays `pick` of the stream,
    repeated until at least `min_seconds` of CPU work are timed."""
    import torch
    from oracle import ora
    threads = host_threads()
    sample = len(pick)
    sub = wrays[:, torch.from_numpy(pick).to(wrays.device)].cpu().numpy()
    w = ora.wrays_from_planes(sub)
    o = ora.OracleScene(scene_py)
    inter = None
    reps = 0
    t0 = time.perf_counter()
    while True:
        inter = o.trace(w, threads=threads, chunk=65536)
        reps += 1
        dt = time.perf_counter() - t0
        if dt >= min_seconds:
            break
    return sample * reps / dt / 1e6, threads, inter, dt, reps


PROFILE = os.path.join(ROOT, "profiles", "trace_heightfield_stream.txt")


def _profile_value(key):
    """A `key: value` figure of the main pass's rocprofv3 summary, or None."""
    if not os.path.exists(PROFILE):
        return None
    with open(PROFILE) as f:
        for line in f:
            if line.startswith(key + ":"):
                return float(line.split(":", 1)[1].strip())
    return None


def traffic_from_profile():
    """HBM bytes per main-pass launch measured with rocprofv3 (FETCH_SIZE and
    WRITE_SIZE, scaled by a plain copy's reading), kept beside the profile
    summary; None when that file is absent."""
    return _profile_value("traffic_bytes_per_launch")


def issue_from_profile():
    """The main pass's instruction-issue figures from the same summary: the
    share of time the SIMDs issue VALU instructions (VALUBusy), the active
    lanes per VALU instruction (VALUUtilization) and the mean resident
    waves per SIMD (MeanOccupancyPerCU / 4)."""
    keys = ("valu_busy_pct", "valu_lane_utilization_pct", "waves_per_simd")
    vals = {k: _profile_value(k) for k in keys}
    if any(v is None for v in vals.values()):
        return None
    vals["waves_per_simd_allowed"] = 5
    vals["source"] = "rocprofv3 --pmc VALUBusy VALUUtilization MeanOccupancyPerCU (profiles/trace_heightfield_stream.txt)"
    return vals


# Hero wavelengths of every render: uniform over the reference's
# [380, 700] nm with 3 more at +80 nm steps wrapped into it
# (color/color.hpp:15-16, 31-38), not the [380, 780] some configurations name.
HERO_WAVELENGTH_NM = [380.0, 700.0]

# names of PSY_RENDER_* and PSY_TRACE_MODE_* (include/psy_gpu.h)
RENDER_FORMS = {0: "wavefront", 1: "fused", 2: "stream"}
TRACE_MODES = {0: "plain", 1: "persistent", 2: "persistent-coherent", 3: "plain-coherent"}

REF_BUCKET_PATHS = 65536   # Config::samples_per_bucket (config.cpp:12; integrator/path_trace_integrator.cpp:29-34)


def _render_rate(gpu, ctx, g, W, H, spp, pl, reps=2):
    """(Mrays/s, film) of psy_render with the context's current settings."""
    import torch
    film, _, rays = gpu.render(ctx, g, W, H, spp, 1, pl)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(reps):
        film, _, rays = gpu.render(ctx, g, W, H, spp, 1, pl)
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / reps
    return rays / dt / 1e6, film


def batching_forms():
    """The batched / autotuned integrator against the plain wavefront: the
    same images (bit-identical samples), Mrays/s of each form."""
    import torch
    from psychopath_cpp_amd import configs, gpu
    out = []
    for name, make, W, H, spp, pl in (
            ("heightfield 64x64 bilinear patches (dice_rate 1.0), 1024x1024, 16 spp, path length 4",
             configs.heightfield_scene, 1024, 1024, 16, 4),
            ("4096 bicubic patches on a sphere instanced 16x (2 levels, 2-sample motion), DoF 0.05, 480x270, "
             "4 spp, path length 6", configs.bicubic_sphere_scene, 480, 270, 4, 6)):
        ctx = gpu.Context(0)
        g = gpu.GpuScene(ctx, make())
        gpu.set_render_mode(ctx)
        gpu.set_render_streams(ctx, 1)
        gpu.set_render_chunk(ctx, REF_BUCKET_PATHS)
        plain, f_plain = _render_rate(gpu, ctx, g, W, H, spp, pl, reps=1)
        log(f"batching [{name[:40]}]: plain wavefront, {REF_BUCKET_PATHS}-path buckets: {plain:.1f} Mrays/s")
        gpu.set_render_streams(ctx, 4)
        gpu.set_render_chunk(ctx, 1 << 21)
        dflt, f_dflt = _render_rate(gpu, ctx, g, W, H, spp, pl)
        log(f"batching: wavefront, library default 2^21-path chunks, four in flight: {dflt:.1f} Mrays/s")
        gpu.set_render_chunk(ctx, 1 << 22)
        wide, f_wide = _render_rate(gpu, ctx, g, W, H, spp, pl)
        log(f"batching: wavefront, 2^22-path chunks, four in flight: {wide:.1f} Mrays/s")
        d0 = int(g.info.dice_depth)
        t0 = time.perf_counter()
        tune = gpu.autotune_render(ctx, g, W, H, spp, path_length=pl)
        tune_s = time.perf_counter() - t0
        tuned, f_tuned = _render_rate(gpu, ctx, g, W, H, spp, pl)
        log(f"batching: autotuned {tune} in {tune_s:.2f} s: {tuned:.1f} Mrays/s")
        # forms give identical images at one dicing depth; a re-diced scene
        # (the tuner's depth) can differ where two micro-patches tie in t
        f_ref = f_plain
        if int(tune["dice_depth"]) != d0:
            ref_ctx = gpu.Context(0)
            f_ref, _, _ = gpu.render(ref_ctx, g, W, H, spp, 1, pl)  # library defaults, the tuned depth
            ref_ctx.close()
        same = bool(torch.equal(f_ref, f_tuned) and torch.equal(f_plain, f_wide) and torch.equal(f_plain, f_dflt))
        depth_rel = float(((f_tuned - f_plain).abs() / (f_plain.abs() + 1e-6)).max())
        out.append({"workload": name, "plain_mrays": round(plain, 2),
                    "plain_form": f"wavefront, {REF_BUCKET_PATHS}-path buckets, host sync per step",
                    "default_wavefront_mrays": round(dflt, 2),
                    "default_form": "wavefront, the library's default 2^21-path chunks, four in flight",
                    "wavefront_2p22_mrays": round(wide, 2), "autotuned_mrays": round(tuned, 2),
                    "autotuned": {"form": RENDER_FORMS.get(int(tune["mode"]), str(tune["mode"])),
                                  "paths": int(tune["pool"]),
                                  "trace": TRACE_MODES.get(int(tune["trace_mode"]), str(tune["trace_mode"])),
                                  "stack": int(tune["stack"]), "steps_per_graph": int(tune["steps_per_graph"]),
                                  "dice_depth": int(tune["dice_depth"]), "scene_dice_depth": d0,
                                  "streams": int(tune["streams"]), "shade_waves": int(tune["shade_waves"]),
                                  "tune_seconds": round(tune_s, 2)},
                    "speedup_vs_plain": round(tuned / plain, 2),
                    "speedup_vs_default_wavefront": round(tuned / dflt, 2),
                    "speedup_vs_2p22_wavefront": round(tuned / wide, 2),
                    "images_identical": same, "film_max_rel_vs_scene_depth": depth_rel,
                    "hero_wavelength_nm": HERO_WAVELENGTH_NM})
        g.close()
        ctx.close()
    return out


def full_config_renders():
    """Renders of the four scene configurations at their own sizes, each
    with the autotuned setting (psy_render_autotune): Mrays/s and ms per
    render.  The lights are RGB (the reference's lights carry an RGB colour;
    C3's two-Gaussian spectra have no counterpart there)."""
    import torch
    from psychopath_cpp_amd import configs, gpu
    out = []
    for name, make, W, H, spp, pl in (
            ("C0 64 spheres + ground, 2 lights, 256x256, 16 spp, path length 4", configs.sphere_scene, 256, 256, 16, 4),
            ("C1 heightfield 64x64 bilinear patches, 1024x1024, 64 spp, path length 4", configs.heightfield_scene,
             1024, 1024, 64, 4),
            ("C2 4096 bicubic patches instanced 16x with motion, DoF, 1920x1080, 32 spp, path length 6",
             configs.bicubic_sphere_scene, 1920, 1080, 32, 6),
            ("C3 sphere scene + 10000 sphere lights, 1024x1024, 64 spp, path length 4", configs.many_light_scene,
             1024, 1024, 64, 4)):
        log(f"full config: {name}")
        ctx = gpu.Context(0)
        g = gpu.GpuScene(ctx, make())
        d0 = int(g.info.dice_depth)
        t0 = time.perf_counter()
        tune = gpu.autotune_render(ctx, g, W, H, spp, path_length=pl)
        tune_s = time.perf_counter() - t0
        rate, film = _render_rate(gpu, ctx, g, W, H, spp, pl, reps=1)
        torch.cuda.synchronize()
        log(f"full config: {rate:.1f} Mrays/s ({tune})")
        out.append({"workload": name, "mrays": round(rate, 1),
                    "autotuned": {"form": RENDER_FORMS.get(int(tune["mode"]), str(tune["mode"])),
                                  "paths": int(tune["pool"]),
                                  "trace": TRACE_MODES.get(int(tune["trace_mode"]), str(tune["trace_mode"])),
                                  "stack": int(tune["stack"]), "dice_depth": int(tune["dice_depth"]),
                                  "scene_dice_depth": d0, "streams": int(tune["streams"]),
                                  "shade_waves": int(tune["shade_waves"])},
                    "tune_seconds": round(tune_s, 2),
                    "film_mean_xyz": [round(float(v), 6) for v in film.mean(dim=(0, 1)).cpu().tolist()]})
        g.close()
        ctx.close()
    return out


def render_profile():
    """One render each of C1 (1024x1024, 16 spp, path length 4) and C2
    (960x540, 8 spp, path length 6) after a warm-up render, with one
    wavefront chunk in flight so that kernel durations do not overlap: the
    integrator's time per kernel under a kernel-trace profiler."""
    import torch
    from psychopath_cpp_amd import configs, gpu
    out = []
    for name, make, W, H, spp, pl, stack, depth in (
            ("C1 heightfield 1024x1024, 16 spp, path length 4", configs.heightfield_scene, 1024, 1024, 16, 4, 16, -1),
            ("C2 bicubic motion 960x540, 8 spp, path length 6", configs.bicubic_sphere_scene, 960, 540, 8, 6, 32, 12)):
        ctx = gpu.Context(0)
        g = gpu.GpuScene(ctx, make(), dice_depth=depth)
        gpu.set_render_mode(ctx)
        ctx.set_trace_mode(persistent=False, coherent=True)
        ctx.set_trace_stack(stack)
        gpu.set_render_streams(ctx, 1)
        gpu.set_render_chunk(ctx, 1 << 23)
        gpu.render(ctx, g, W, H, spp, 1, pl)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        _, _, rays = gpu.render(ctx, g, W, H, spp, 1, pl)
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
        log(f"render profile [{name}]: {rays} rays in {dt * 1e3:.2f} ms")
        out.append({"workload": name, "rays": int(rays), "ms": round(dt * 1e3, 2),
                    "mrays": round(rays / dt / 1e6, 1), "dice_depth": int(g.info.dice_depth)})
        g.close()
        ctx.close()
    return out


def subdivision_stream(args):
    """The primary + first-bounce stream (2^21 + 2^21 rays) through the
    Catmull-Clark scene (configs.subdivision_scene: the heightfield as one
    control mesh, 25 instanced rounded boxes): trace Mrays/s with the main
    and second pass timed by HIP events, the host's patch extraction, and
    the oracle on a sample of the same rays.  Each step is one
    psy_trace_world call (world rays in, closest hits out)."""
    import numpy as np
    import torch
    from oracle import ora
    from psychopath_cpp_amd import configs, gpu
    scene_py = configs.subdivision_scene()
    field = scene_py.root.objects[0]
    t0 = time.perf_counter()
    reps = 0
    while time.perf_counter() - t0 < 0.5 or reps < 3:
        patches = gpu.subdivision_patches(field.data, field.face_vert_counts, field.face_vert_indices)
        reps += 1
    extract_ms = (time.perf_counter() - t0) / reps * 1e3
    t0 = time.perf_counter()
    reps = 0
    while time.perf_counter() - t0 < 0.5 or reps < 3:
        ora.subdiv_patches(field.data, field.face_vert_counts, field.face_vert_indices)
        reps += 1
    ora_extract_ms = (time.perf_counter() - t0) / reps * 1e3
    ctx = gpu.Context(0)
    if args.continuation is not None:
        ctx.set_continuation(args.continuation)
    t0 = time.perf_counter()
    g = gpu.GpuScene(ctx, scene_py, dice_depth=args.dice_depth)
    torch.cuda.synchronize()
    build_s = time.perf_counter() - t0
    info = g.info
    log(f"subdivision scene: {len(patches)} field patches ({extract_ms:.2f} ms to extract), "
        f"{info.n_leaf_instances} leaves, dice depth {info.dice_depth}, built in {build_s:.2f}s")
    wrays, n_valid = make_stream(ctx, g)
    # the boxes are transformed patch instances: their ray footprints come
    # from world rays (psy_trace_world, Tracer::trace's own interface)
    hits = gpu.HitBuffers(STREAM_RAYS, wrays.device, aux=False)
    for _ in range(args.warmup):
        gpu.trace_world(ctx, g, wrays, hits=hits)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream()
    ev0 = torch.cuda.Event(enable_timing=True)
    ev1 = torch.cuda.Event(enable_timing=True)
    ctx.set_trace_timing(True)
    ctx.trace_timing()
    ev0.record(stream)
    for _ in range(args.steps):
        gpu.trace_world(ctx, g, wrays, hits=hits)
    ev1.record(stream)
    torch.cuda.synchronize()
    main_ms, second_ms, calls = ctx.trace_timing()
    ctx.set_trace_timing(False)
    ms = ev0.elapsed_time(ev1) / args.steps
    mrays = STREAM_RAYS / (ms / 1e3) / 1e6
    log(f"subdivision stream: {ms:.3f} ms/step = {mrays:.1f} Mrays/s; main {main_ms / max(calls, 1):.3f} ms, "
        f"second {second_ms / max(calls, 1):.3f} ms per call, {ctx.retrace_count()} rays in the second pass")
    out = {"workload": "subdivision_scene: 64x64-quad Catmull-Clark heightfield + 25 rounded boxes, "
                       "2^21 primary + 2^21 bounce rays",
           "field_patches": len(patches), "leaves": int(info.n_leaf_instances), "dice_depth": int(info.dice_depth),
           "extract_ms": round(extract_ms, 2), "oracle_extract_ms": round(ora_extract_ms, 2),
           "scene_build_s": round(build_s, 3), "ms_per_step": round(ms, 4), "mrays": round(mrays, 1),
           "main_pass_ms": round(main_ms / max(calls, 1), 4), "second_pass_ms": round(second_ms / max(calls, 1), 4),
           "second_pass_rays": int(ctx.retrace_count()), "valid_bounces": n_valid}
    if not args.no_cpu:
        sample = min(args.cpu_sample, STREAM_RAYS)
        pick = mixed_sample(STREAM_RAYS, sample)
        cpu_mrays, threads, inter, dt, reps = cpu_baseline(scene_py, wrays, pick, args.cpu_seconds)
        ids = g.instance_ids()
        tp = torch.from_numpy(pick).to(hits.inst.device)
        gi = hits.inst[tp].cpu().numpy().view(np.uint32)
        gt = hits.t[tp].cpu().numpy()
        ghit = gi != 0xFFFFFFFF
        ok = ghit == (inter["hit"] != 0)
        both = ghit & (inter["hit"] != 0)
        ok[both] &= ids[gi[both]] == inter["id"][both]
        ok[both] &= np.abs(gt[both] - inter["t"][both]) <= 1e-5 * np.abs(inter["t"][both])
        log(f"subdivision cpu baseline: {cpu_mrays:.3f} Mrays/s on {threads} threads; parity {ok.mean():.6f}")
        out["cpu_baseline"] = {"value": round(cpu_mrays, 4), "unit": "Mrays/s", "cores": threads, "kind": "port",
                               "sample": f"{sample} rays of the stream (half primary, half bounce), {reps} passes"}
        out["parity_on_cpu_sample"] = round(float(ok.mean()), 6)
    g.close()
    ctx.close()
    return out


def adjoint_timing():
    """Adjoint / forward time of the differentiable render."""
    import numpy as np
    import torch
    from psychopath_cpp_amd import configs, gpu
    ctx = gpu.Context(0)
    sc = configs.adjoint_scene()
    g = gpu.GpuScene(ctx, sc)
    rng = np.random.default_rng(1)
    alb0, _ = g.get_params()
    n_l = g.param_counts()[1]
    target, _, _ = gpu.render(ctx, g, 512, 512, 16, 1)
    g.set_params((alb0 * rng.uniform(0.5, 1.5, alb0.size)).astype(np.float32),
                 rng.uniform(0.5, 1.5, n_l).astype(np.float32))
    film, _, _ = gpu.render(ctx, g, 512, 512, 16, 1)
    d = (2.0 * (film - target)).float().contiguous()
    gpu.adjoint(ctx, g, d, 16, 1)
    torch.cuda.synchronize()
    reps = 5
    t0 = time.perf_counter()
    for _ in range(reps):
        gpu.render(ctx, g, 512, 512, 16, 1)
    torch.cuda.synchronize()
    tf = (time.perf_counter() - t0) / reps
    t0 = time.perf_counter()
    for _ in range(reps):
        gpu.adjoint(ctx, g, d, 16, 1)
    torch.cuda.synchronize()
    ta = (time.perf_counter() - t0) / reps
    log(f"adjoint: forward {tf * 1e3:.2f} ms, adjoint {ta * 1e3:.2f} ms, ratio {ta / tf:.2f}")
    g.close()
    ctx.close()
    return {"workload": "256 spheres + ground, 1000 sphere lights, 512x512, 16 spp, path length 4; gradients of an "
                        "L2 image loss w.r.t. 257 albedos and 1000 emission scales",
            "forward_ms": round(tf * 1e3, 3), "adjoint_ms": round(ta * 1e3, 3), "ratio": round(ta / tf, 3),
            "hero_wavelength_nm": HERO_WAVELENGTH_NM}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--cpu-sample", type=int, default=1 << 21)
    ap.add_argument("--cpu-seconds", type=float, default=10.0, help="minimum CPU baseline time (repeats the sample)")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-forms", action="store_true", help="skip the batching and adjoint measurements")
    ap.add_argument("--full-configs", action="store_true",
                    help="only render the four scene configurations at their own sizes (autotuned) and print them")
    ap.add_argument("--subdiv", action="store_true",
                    help="only time the ray stream through the Catmull-Clark scene (configs.subdivision_scene)")
    ap.add_argument("--dice-depth", type=int, default=-1)
    ap.add_argument("--trace-mode", choices=("persistent", "plain"), default="plain",
                    help="main trace pass: persistent waves with lane refill, or one thread per ray")
    ap.add_argument("--refill", type=int, default=16, help="persistent mode: refill a wave once this many lanes idle")
    ap.add_argument("--continuation", type=int, default=None,
                    help="plain mode: a wave hands its rays to a follow-on launch once fewer than this many trace "
                         "(0: never; default: the library's, 24 for object rays and never for world rays)")
    ap.add_argument("--blocks-per-cu", type=int, default=0, help="persistent mode: blocks per CU (0: occupancy)")
    ap.add_argument("--split", action="store_true",
                    help="also time the primary and the bounce half of the stream separately (stderr)")
    ap.add_argument("--render-profile", action="store_true",
                    help="only render C1 (1024x1024x16) and C2 (960x540x8) once each with one wavefront chunk in "
                         "flight, for a per-kernel profile of the integrator")
    ap.add_argument("--copy-probe", type=int, default=0, metavar="BYTES",
                    help="only run a plain device-to-device copy of BYTES (calibrates rocprofv3 byte counters)")
    args = ap.parse_args()
    if args.full_configs:
        print(json.dumps({"full_config_renders": full_config_renders()}), flush=True)
        return 0
    if args.subdiv:
        print(json.dumps({"subdivision_stream": subdivision_stream(args)}), flush=True)
        return 0
    if args.render_profile:
        print(json.dumps({"render_profile": render_profile()}), flush=True)
        return 0
    if args.copy_probe:
        import torch
        src = torch.empty(args.copy_probe // 4, dtype=torch.float32, device="cuda").fill_(1.0)
        dst = torch.empty_like(src)
        torch.cuda.synchronize()
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        log(f"copy probe: 3 copies of {args.copy_probe} bytes")
        return 0
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported (every box has one GPU; "
              "the path would shard by image tiles or ray ranges)", file=sys.stderr)
        return 2

    import torch
    from psychopath_cpp_amd import configs, gpu

    log("setting up heightfield scene")
    ctx = gpu.Context(0)
    if args.continuation is not None:
        ctx.set_continuation(args.continuation)
    ctx.set_trace_mode(persistent=args.trace_mode == "persistent", refill_min=args.refill,
                       blocks_per_cu=args.blocks_per_cu)
    scene_py = configs.heightfield_scene()
    t0 = time.perf_counter()
    scene = gpu.GpuScene(ctx, scene_py, dice_depth=args.dice_depth)
    torch.cuda.synchronize()
    build_s = time.perf_counter() - t0
    info = scene.info
    log(f"scene: {info.n_leaf_instances} leaves, {info.n_bvh_nodes} BVH4 nodes, dice depth {info.dice_depth}, "
        f"{info.dice_cache_bytes / 2**20:.0f} MiB dice cache, built in {build_s:.2f}s")
    wrays, n_valid = make_stream(ctx, scene)
    rays = gpu.world_to_rays(ctx, wrays)
    hits = gpu.HitBuffers(STREAM_RAYS, rays.device, aux=False)
    torch.cuda.synchronize()
    log(f"stream: {rays.shape[1]} rays ({n_valid} valid bounces)")

    for _ in range(args.warmup):
        gpu.trace_rays(ctx, scene, rays, hits=hits)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream()
    ev0 = torch.cuda.Event(enable_timing=True)
    ev1 = torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    # the library records HIP events on its launch stream around the main
    # pass (the dominant kernel) and the second pass of every trace call
    ctx.set_trace_timing(True)
    ctx.trace_timing()
    t_wall = time.perf_counter()
    ev0.record(stream)
    for _ in range(args.steps):
        gpu.trace_rays(ctx, scene, rays, hits=hits)
    ev1.record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t_wall
    main_ms, second_ms, calls = ctx.trace_timing()
    ctx.set_trace_timing(False)
    ms = ev0.elapsed_time(ev1) / args.steps
    mrays = STREAM_RAYS / (ms / 1e3) / 1e6
    main_avg = main_ms / max(calls, 1)
    achieved = BYTES_PER_RAY * STREAM_RAYS / (main_avg / 1e3) / 1e9
    hit_frac = float((hits.inst != -1).float().mean().item())
    log(f"trace ({args.trace_mode}): {ms:.3f} ms/step (HIP events), wall {wall / args.steps * 1e3:.3f} ms/step, "
        f"hit fraction {hit_frac:.4f}, second pass {ctx.retrace_count()} rays")
    log(f"passes over {calls} calls: main {main_avg:.3f} ms/launch, second {second_ms / max(calls, 1):.3f} ms/launch")

    if args.split:
        half = STREAM_RAYS // 2
        for name, sl in (("primary", slice(0, half)), ("bounce", slice(half, STREAM_RAYS))):
            sub = rays[:, sl].contiguous()
            hs = gpu.HitBuffers(half, rays.device, aux=False)
            gpu.trace_rays(ctx, scene, sub, hits=hs)
            torch.cuda.synchronize()
            ev0.record(stream)
            for _ in range(args.steps):
                gpu.trace_rays(ctx, scene, sub, hits=hs)
            ev1.record(stream)
            torch.cuda.synchronize()
            pms = ev0.elapsed_time(ev1) / args.steps
            log(f"split {name}: {pms:.3f} ms for {half} rays = {half / (pms / 1e3) / 1e6:.1f} Mrays/s, "
                f"second pass {ctx.retrace_count()} rays")

    cpu = None
    if not args.no_cpu:
        sample = min(args.cpu_sample, STREAM_RAYS)
        pick = mixed_sample(STREAM_RAYS, sample)
        model = cpu_model()
        log(f"cpu baseline: oracle breadth-first tracer on {sample} rays (half primary, half bounce), {model}")
        cpu_mrays, threads, inter, dt, reps = cpu_baseline(scene_py, wrays, pick, args.cpu_seconds)
        log(f"cpu baseline: {cpu_mrays:.3f} Mrays/s on {threads} threads ({reps} passes, {dt:.1f}s)")
        # spot parity on the same sample
        import numpy as np
        ids = scene.instance_ids()
        tp = torch.from_numpy(pick).to(hits.inst.device)
        gi = hits.inst[tp].cpu().numpy().view(np.uint32)
        gt = hits.t[tp].cpu().numpy()
        ghit = gi != 0xFFFFFFFF
        ok = (ghit == (inter["hit"] != 0))
        both = ghit & (inter["hit"] != 0)
        ok[both] &= ids[gi[both]] == inter["id"][both]
        ok[both] &= np.abs(gt[both] - inter["t"][both]) <= 1e-5 * np.abs(inter["t"][both])
        log(f"parity on the cpu sample: {ok.mean():.6f} of rays match")
        cpu = {"value": round(cpu_mrays, 4), "unit": "Mrays/s", "cores": threads, "kind": "port",
               "cpu_model": model,
               "host_cpus": os.cpu_count(),
               "sample": f"{sample} rays of the same 2^22 stream, an equal mix of its two halves (the first "
                         f"{sample // 2} primary rays, 1024x1024x2 spp, and the first {sample - sample // 2} "
                         f"cosine first-bounce rays), traced {reps} times ({dt:.1f} s) by the oracle restatement "
                         f"of the reference breadth-first BVH4 + split-dice tracer, 65536-ray chunks, "
                         f"{threads} threads (this process's CPU affinity, capped by OMP_NUM_THREADS)"}

    out = {
        "metric": METRIC,
        "value": round(mrays, 2),
        "unit": "Mrays/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": "heightfield 64x64 bilinear patches over 10x10 (8 seeded sines), dice_rate 1.0; "
                        "2^22-ray closest-hit stream = 2^21 primary (1024x1024, 2 spp) + 2^21 cosine first-bounce",
            "rays_per_step": STREAM_RAYS,
            "dice_depth": int(info.dice_depth),
            "leaf_instances": int(info.n_leaf_instances),
            "bytes_per_ray": BYTES_PER_RAY,
            "trace_mode": args.trace_mode,
            "continuation_below": 24 if args.continuation is None else args.continuation,
        },
        "roofline": {
            "kernel": "k_trace<false, 16, false> + k_trace_cont<false, 16> (main pass, %.3f ms/call)" % main_avg,
            "bound": "hbm",
            "achieved": round(achieved, 2),
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 5),
            "traffic": traffic_from_profile(),
            "issue": issue_from_profile(),
        },
        "cpu_baseline": cpu,
    }
    if not args.no_forms:
        out["batching"] = batching_forms()
        out["adjoint"] = adjoint_timing()
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
