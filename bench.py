#!/usr/bin/env python3
"""Particle-updates/s of the position-based-fluids substep on one MI355X.

Default workload (the 8M-particle configuration of the headline metric):
double dam break, two 256x128x128 FP32 lattice blocks (8,388,608 particles),
spacing s = 0.008 m, seeded +-0.01 s jitter, at the two x-ends of a 6x2x2 m box;
h = 2s, rho0 = 1000, mass rho0 s^3, dt = 1/300 s, g = 9.81, relaxation 600,
4 Jacobi iterations, surface tension 0.5, vorticity confinement 0.01
(m/rho-weighted form), XSPH 0.01, and a torus (R 0.4, r 0.12) united with an
axis-aligned box, sampled onto a 256^3 FP32 SDF grid.

One step = one substep of the solver over all particles with the state
resident in HBM, replayed from a captured HIP graph (--no-graph: eager
launches).  Prints one JSON line: the throughput, the roofline of the dominant
kernel (the same substeps launched eagerly, every kernel event-timed on the
library's stream), the VALU floor of each gather kernel (VALU instructions per
launch from the committed rocprofv3 SQ_INSTS_VALU summary), Jacobi iterations
and error to 0.1% density error in
tolerance mode, plain and warm-started (trained network file), and the FP64
CPU oracle timed on the host cores on a bounded sample of the same state
(reported baseline only).  --workload batch times the batched-scene workload.
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

METRIC = "particle-updates/s @8M; Jacobi iters to 0.1% density err, warm-start vs plain"
HBM_PEAK_GBS = 8000.0

# Algorithmic bytes per particle of each kernel (FP32, each stream once per
# pass, 3-vectors 12 B, scalars 4 B, a neighbour list 4(nbar+1) B).
VALU_SIMDS = 256 * 4        # MI355X: 256 CUs x 4 SIMDs
VALU_CLOCK_HZ = 2.4e9       # peak engine clock
KERNEL_BYTES = {
    "density_lambda": lambda L: 20 + L,   # x* 12, list -> rho 4, lambda 4
    "dp_update": lambda L: 28 + L,        # x* 12, lambda 4, list -> x*' 12
    "build_lists": lambda L: 12 + L,      # x* 12 -> list
    "color": lambda L: 64 + L,            # velocity (x*, x -> v) + colour (x*, rho -> n)
    "surface": lambda L: 52 + L,          # x*, rho, n, v -> v
    "xsph": lambda L: 40 + L,             # x*, rho, v -> v
    "vorticity": lambda L: 40 + L,        # x*, v -> omega
    "confine": lambda L: 68 + L,          # x*, omega, v, id -> x, v (commit)
}


def scene_double_dam_break(scale=1.0):
    from sphpc_amd import workloads
    return workloads.double_dam_break(scale)


def gpu_params(sc, iters=4, tol=0.0):
    import sphpc_amd as sa
    s = sc["s"]
    return sa.default_params(2.0 * s, time_step=1.0 / 300.0, g=9.81, k=0.5, c=0.01,
                             rest_density=1000.0, rest_mass=1000.0 * s ** 3,
                             lambda_epsilon=600.0, vorticity_epsilon=0.01, vorticity_model=1,
                             solve_iterations=iters, density_tolerance=tol)


def read_traffic(kernel, workload_tag):
    """HBM bytes per launch from the committed rocprofv3 --pmc summary, or None."""
    path = os.path.join(ROOT, "profiles", f"pmc_traffic_{workload_tag}.txt")
    if not os.path.exists(path):
        return None
    for line in open(path):
        parts = line.split()
        if parts and parts[0] == kernel:
            for tok in parts[1:]:
                if tok.startswith("bytes_per_launch="):
                    return float(tok.split("=", 1)[1])
    return None


def read_valu(kernel, workload_tag):
    """VALU instructions per launch from the committed rocprofv3 --pmc summary, or None."""
    path = os.path.join(ROOT, "profiles", f"pmc_valu_{workload_tag}.txt")
    if not os.path.exists(path):
        return None
    for line in open(path):
        parts = line.split()
        if parts and parts[0] == kernel:
            for tok in parts[1:]:
                if tok.startswith("valu_insts_per_launch="):
                    return float(tok.split("=", 1)[1])
    return None


def valu_ceiling(times, n, nbar, tag):
    """Per gather kernel: the time its VALU instructions take at full issue rate
    (wave64 instructions x 4 cycles over 1024 SIMDs at 2.4 GHz; a lower bound,
    transcendentals issue at quarter rate), against its measured launch time, and
    the HBM roofline fraction the kernel would reach at that VALU floor.  Where
    that fraction is below 0.6 the 60% target is out of reach for the kernel."""
    L = 4.0 * (nbar + 1.0)
    out = {}
    for k, (ms, cnt) in times.items():
        if k not in KERNEL_BYTES:
            continue
        insts = read_valu(k, tag)
        if insts is None:
            continue
        floor_s = insts * 4.0 / (VALU_SIMDS * VALU_CLOCK_HZ)
        frac = KERNEL_BYTES[k](L) * n / floor_s / (HBM_PEAK_GBS * 1e9)
        out[k] = {"valu_insts_per_launch": insts, "valu_floor_ms": floor_s * 1e3,
                  "avg_launch_ms": ms / cnt, "valu_busy": floor_s * 1e3 / (ms / cnt),
                  "hbm_frac_at_valu_floor": frac, "target_0p6_out_of_reach": frac < 0.6}
    return out


def cpu_baseline(sc, substeps, threads):
    """FP64 oracle (C, OpenMP) on the same initial state: 1 warm-up substep, then
    `substeps` timed ones.  Reported baseline only."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import orc
    os.environ.setdefault("OMP_NUM_THREADS", str(threads))
    L = orc.oracle()
    p = orc.make_params(sc["s"], sc["box"], dt=1.0 / 300.0, g=9.81, k=0.5, c=0.01,
                        lambda_eps=600.0, vort_eps=0.01, vort_model=1, surface=True,
                        viscosity=True, vorticity=True)
    ob = orc.obstacle(sc["sdf"], sc["dims"], sc["dx"], sc["wmin"], sc["wmax"])
    pos = sc["pos"]
    n = len(pos)
    cols = [np.ascontiguousarray(pos[:, i], dtype=np.float64) for i in range(3)]
    arrs = dict(x=cols[0], y=cols[1], z=cols[2], vx=np.zeros(n), vy=np.zeros(n),
                vz=np.zeros(n), xs=np.zeros(n), ys=np.zeros(n), zs=np.zeros(n),
                density=np.zeros(n), lambda_=np.zeros(n),
                nbr=np.zeros(n * orc.MAXN, np.uint32), cnt=np.zeros(n, np.int32))
    st = orc.OrcState(**{k: v.ctypes.data for k, v in arrs.items()})
    L.orc_set_threads(threads)
    L.orc_substep(n, C.byref(st), C.byref(p), C.byref(ob), 4, 0.0, None)
    t0 = time.perf_counter()
    for _ in range(substeps):
        L.orc_substep(n, C.byref(st), C.byref(p), C.byref(ob), 4, 0.0, None)
    dt = time.perf_counter() - t0
    # one thread (the reference's own CPU path is sequential), one substep of
    # the first 2^20 particle ids of the same initial state
    n1 = min(n, 1 << 20)
    a1 = {k: (np.ascontiguousarray(v[:n1 * orc.MAXN]) if k == "nbr" else
              np.ascontiguousarray(v[:n1])) for k, v in arrs.items()}
    for k, v in zip(("x", "y", "z"), cols):
        a1[k] = np.ascontiguousarray(v[:n1])
    for k in ("vx", "vy", "vz"):
        a1[k] = np.zeros(n1)
    st1 = orc.OrcState(**{k: v.ctypes.data for k, v in a1.items()})
    L.orc_set_threads(1)
    t1 = time.perf_counter()
    L.orc_substep(n1, C.byref(st1), C.byref(p), C.byref(ob), 4, 0.0, None)
    dt1 = time.perf_counter() - t1
    L.orc_set_threads(threads)
    return dict(value=n * substeps / dt, unit="particle-updates/s", cores=threads, kind="port",
                one_thread_value=n1 / dt1,
                sample=f"FP64 C oracle (OpenMP) on the same {n}-particle initial state: "
                       f"1 warm-up + {substeps} timed substeps on {threads} threads ({dt:.1f} s); "
                       f"one_thread_value: 1 substep of its first {n1} particles on 1 thread "
                       f"({dt1:.1f} s); reported baseline only")


def timed_region(ctx, steps):
    """Times `steps` fused substeps; every kernel launch is bracketed by HIP
    events on the library's own stream, whose sums give per-kernel averages."""
    import sphpc_amd as sa
    ctx.synchronize()
    ctx.profile(True)
    ctx.profile_reset()
    t0 = time.perf_counter()
    ctx.step(steps)
    ctx.synchronize()
    elapsed = time.perf_counter() - t0
    times = {}
    for k, name in enumerate(sa.kernel_names()):
        ms, cnt = ctx.profile_read(k)
        if cnt:
            times[name] = (ms, cnt)
    ctx.profile(False)
    return elapsed, times


def roofline(times, n, nbar, steps, tag):
    """Roofline object of the dominant gather kernel plus per-kernel ms per substep."""
    gathers = {k: v for k, v in times.items() if k in KERNEL_BYTES}
    dom = max(gathers, key=lambda k: gathers[k][0])
    ms, cnt = gathers[dom]
    avg_s = ms / cnt / 1e3
    L = 4.0 * (nbar + 1.0)
    bytes_launch = KERNEL_BYTES[dom](L) * n
    achieved = bytes_launch / avg_s / 1e9
    roof = {"bound": "hbm", "kernel": dom, "achieved": achieved, "peak": HBM_PEAK_GBS,
            "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS, "traffic": read_traffic(dom, tag),
            "algorithmic_bytes_per_launch": bytes_launch, "avg_launch_ms": avg_s * 1e3,
            "launches": cnt}
    per = {k: v[0] / steps for k, v in sorted(times.items(), key=lambda kv: -kv[1][0])}
    per["_sum"] = sum(v[0] for v in times.values()) / steps
    return roof, per


GATHER_KERNELS = ("build_lists", "density_lambda", "dp_update", "color", "surface", "xsph",
                  "vorticity", "confine")


def compact_tuning(t):
    if t is None:
        return None
    return {"ms_per_substep_default": t["ms_per_substep_default"],
            "ms_per_substep_tuned": t["ms_per_substep_tuned"],
            "split_collide": t["split_collide"],
            "list_format": "wide" if t["wide_lists"] else "compact",
            "by_rule": [k for k in GATHER_KERNELS if k in t["by_rule"]],
            "threads_per_block": {k: t["block"][k] for k in GATHER_KERNELS},
            "gathers_in_flight": {k: t["depth"][k] for k in GATHER_KERNELS if k != "build_lists"}}


def _err_summary(errs):
    return {"mean": float(np.mean(errs)), "median": float(np.median(errs)),
            "max": float(np.max(errs))}


def run_batch(scenes_count, steps, warmup, graph=True, autotune=True, net_path=None):
    """Batched scenes: `scenes_count` independent scenes in one context, one
    launch per stage for all of them (sphpc_amd/workloads.py), 4 Jacobi
    iterations.  Times `steps` graph-replayed substeps plain and, with a
    network file, the same substeps from the same state warm-started (the
    first iteration's multiplier from the network, plain fallback per scene).
    Returns the result dict."""
    import sphpc_amd as sa
    from sphpc_amd import workloads
    s, scenes, pos = workloads.batched_scenes(scenes_count, seed=4)
    n = len(pos)
    p = sa.default_params(2.0 * s, time_step=1.0 / 300.0, g=9.81, k=0.5, c=0.01,
                          rest_density=1000.0, rest_mass=1000.0 * s ** 3, lambda_epsilon=600.0,
                          vorticity_epsilon=0.01, vorticity_model=1, solve_iterations=4)
    ctx = sa.BatchContext(p, scenes)
    ctx.upload(pos)
    ctx.step(warmup)
    ctx.synchronize()
    tuning = ctx.autotune(3) if autotune else None
    start = ctx.download()

    def timed(warm_net):
        ctx.upload(*start)
        ctx.set_warm_start(warm_net)
        ctx.set_graph(graph)
        ctx.step(1)  # capture (untimed)
        ctx.upload(*start)
        ctx.synchronize()
        t0 = time.perf_counter()
        worst = np.zeros(len(scenes))
        fallbacks = 0
        for _ in range(steps):
            ctx.step(1)
            worst = np.maximum(worst, ctx.scene_errors())
            fallbacks += ctx.stats().warm_fallback
        ctx.synchronize()
        el = time.perf_counter() - t0
        ctx.set_graph(False)
        ctx.set_warm_start(None)
        return el, worst, fallbacks

    # rate without per-substep host reads, then per-scene errors substep by substep
    ctx.upload(*start)
    ctx.set_graph(graph)
    ctx.step(1)
    ctx.upload(*start)
    ctx.synchronize()
    t0 = time.perf_counter()
    ctx.step(steps)
    ctx.synchronize()
    elapsed = time.perf_counter() - t0
    ctx.set_graph(False)
    _, worst_plain, _ = timed(None)
    warm = None
    if net_path and os.path.exists(net_path):
        net = sa.Mlp()
        net.load(net_path)
        el_w, worst_warm, fb = timed(net)
        warm = {"particle_updates_per_s_with_error_reads": n * steps / el_w,
                "scene_max_density_error": _err_summary(worst_warm),
                "scenes_better_than_plain": int(np.sum(worst_warm < worst_plain)),
                "substeps_with_a_fallback": int(fb),
                "network": os.path.relpath(net_path, ROOT)}
    ctx.upload(*start)
    st = ctx.stats()
    prof_steps = max(2, steps // 5)
    _, times = timed_region(ctx, prof_steps)
    nbar = ctx.stats().neighbor_pairs / max(n, 1)
    roof, per = roofline(times, n, nbar, prof_steps, f"pbf_substep_batch{scenes_count}")
    counts = [sc["particles"] for sc in scenes]
    ctx.close()
    return {
        "metric": f"particle-updates/s, {scenes_count} batched scenes",
        "value": n * steps / elapsed, "unit": "particle-updates/s", "n_gpus": 1,
        "steps": steps, "warmup": warmup, "ms_per_step": 1e3 * elapsed / steps,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": f"{scenes_count} independent seeded scenes (2k-128k particles, "
                               "box aspect 1-4, fill 0.1-0.5, sphere SDF 64^3), s=0.01 m, "
                               "4 Jacobi iterations, surface tension + XSPH + vorticity",
                   "particles": n, "scenes": scenes_count, "min_scene": int(min(counts)),
                   "max_scene": int(max(counts)), "graph": graph,
                   "autotune": compact_tuning(tuning), "mean_neighbors": nbar,
                   "neighbor_overflow": st.neighbor_overflow},
        "scene_max_density_error_plain": _err_summary(worst_plain),
        "warm_start": warm,
        "roofline": roof, "kernels_ms_per_substep_eager": per,
    }


def bench_batch(args):
    out = run_batch(args.scenes, args.steps, args.warmup, graph=not args.no_graph,
                    autotune=not args.no_autotune, net_path=args.batch_net)
    print(json.dumps(out), flush=True)


def later_window(ctx, start, first, count, graph):
    """Throughput over substeps [first, first + count) of the run, replayed
    from the state saved at `first` (the fused substep from `start`, the state
    at substep `start_at`)."""
    ctx.upload(*start[1])
    ctx.set_graph(False)
    if first > start[0]:
        ctx.step(first - start[0])
    saved = ctx.download()
    ctx.set_graph(graph)
    ctx.step(1)
    ctx.upload(*saved)
    ctx.synchronize()
    t0 = time.perf_counter()
    ctx.step(count)
    ctx.synchronize()
    el = time.perf_counter() - t0
    ctx.set_graph(False)
    st = ctx.stats()
    n = ctx.count()
    return {"substeps": [first, first + count], "value": n * count / el,
            "ms_per_step": 1e3 * el / count,
            "mean_neighbors": st.neighbor_pairs / max(n, 1),
            "max_density_error_last": st.max_density_error,
            "neighbor_overflow_last": st.neighbor_overflow}


def main():
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--scale", type=float, default=1.0,
                    help="block edge scale (1.0 = the 8,388,608-particle workload)")
    ap.add_argument("--tol-steps", type=int, default=10)
    ap.add_argument("--cpu-steps", type=int, default=3)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-extras", action="store_true",
                    help="only the timed substeps (for profiler runs)")
    ap.add_argument("--net", default=os.path.join(ROOT, "sphpc_amd", "data", "warm_net_s0.008.bin"),
                    help="trained warm-start network (sphpc_amd/warm_train.py)")
    ap.add_argument("--workload", choices=["dam8m", "batch"], default="dam8m",
                    help="dam8m: the 8M double dam break (the headline line); "
                         "batch: independent batched scenes")
    ap.add_argument("--scenes", type=int, default=512)
    ap.add_argument("--no-graph", action="store_true",
                    help="eager launches instead of a captured graph in the timed region")
    ap.add_argument("--no-autotune", action="store_true",
                    help="default launch configuration instead of the autotuner's")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="first run two 1 GiB device copies (counter calibration)")
    ap.add_argument("--batch-net", default=os.path.join(ROOT, "sphpc_amd", "data",
                                                        "warm_net_s0.008.bin"),
                    help="network for the warm-started batch run ('' for none)")
    ap.add_argument("--prev-scale", type=float, default=0.5,
                    help="scale of the previous-multiplier warm start (0: not run)")
    ap.add_argument("--eq-steps", type=int, default=5,
                    help="substeps per iteration count in the equal-accuracy comparison")
    ap.add_argument("--batch-steps", type=int, default=20,
                    help="substeps of the batched-scene run of the default line")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only (asked for {args.gpus}); "
              "the multi-GPU slab decomposition is design-only", file=sys.stderr)
        sys.exit(2)

    import sphpc_amd as sa

    if args.calibrate_copy:
        # a plain copy of known size, so hardware byte counters can be scaled
        nbytes = 1 << 30
        src, dst = sa.DeviceBuffer(nbytes), sa.DeviceBuffer(nbytes)
        for _ in range(2):
            sa.check(sa.lib().sph_device_copy(dst.ptr, src.ptr, nbytes, None))
        src.free()
        dst.free()

    if args.workload == "batch":
        bench_batch(args)
        return

    sc = scene_double_dam_break(args.scale)
    n = len(sc["pos"])
    ctx = sa.Context(gpu_params(sc), sc["box"], n)
    ctx.upload(sc["pos"])
    ctx.set_obstacle(sc["sdf"], sc["dims"], sc["dx"], sc["wmin"], sc["wmax"])

    ctx.step(args.warmup)
    ctx.synchronize()
    tuning = None if args.no_autotune else ctx.autotune(3)
    start = ctx.download()
    start_at = args.warmup
    # Whole-job throughput: substeps replayed from a captured HIP graph (the
    # capture happens during the first, untimed call), state resident in HBM,
    # no per-kernel events in the timed region.
    ctx.set_graph(not args.no_graph)
    ctx.step(1)
    ctx.upload(*start)
    ctx.synchronize()
    t0 = time.perf_counter()
    ctx.step(args.steps)
    ctx.synchronize()
    elapsed = time.perf_counter() - t0
    ctx.set_graph(False)
    # Per-kernel durations: the first substeps of the timed region again, from
    # the same state, launched eagerly with every kernel bracketed by HIP
    # events on the library's stream.
    ctx.upload(*start)
    prof_steps = min(args.steps, 20)
    _, times = timed_region(ctx, prof_steps)
    value = n * args.steps / elapsed
    st = ctx.stats()
    nbar = st.neighbor_pairs / max(n, 1)
    out = {
        "metric": METRIC, "value": value, "unit": "particle-updates/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": 1e3 * elapsed / args.steps,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": "double dam break: 2x256x128x128 FP32 lattice blocks, s=0.008 m, "
                               "6x2x2 m box, torus+box SDF 256^3, 4 Jacobi iterations, "
                               "surface tension + XSPH + vorticity",
                   "particles": n, "scale": args.scale, "mean_neighbors": nbar,
                   "max_density_error_last": st.max_density_error,
                   "neighbor_overflow": st.neighbor_overflow},
    }
    out["roofline"], out["kernels_ms_per_substep"] = roofline(
        times, n, nbar, prof_steps, "pbf_substep_8M" if args.scale == 1.0 else f"pbf_substep_scale{args.scale}")
    out["valu_ceiling"] = valu_ceiling(
        times, n, nbar, "pbf_substep_8M" if args.scale == 1.0 else f"pbf_substep_scale{args.scale}")
    out["config"]["graph"] = not args.no_graph
    out["config"]["autotune"] = compact_tuning(tuning)
    if not args.no_extras:
        # Jacobi iterations and wall time to max density error <= 0.1% (cap 10),
        # plain and warm-started, from the same state (the state after the
        # timed substeps); the warm start needs a trained network file.
        from sphpc_amd import warm_train
        pos, vel = ctx.download()
        tol_params = gpu_params(sc, iters=10, tol=1e-3)
        net = None
        if os.path.exists(args.net):
            net = sa.Mlp()
            net.load(args.net)
        if net is not None:
            cmp = warm_train.compare(ctx, net, pos, vel, tol_params, args.tol_steps,
                                     log=lambda m: print(m, file=sys.stderr),
                                     prev_scale=args.prev_scale)
        else:
            ctx.upload(pos, vel)
            ctx.set_params(tol_params)
            cmp = {"plain": None, "warm": None}
            its, errs, t_el = [], [], 0.0
            ctx.step(1)
            for _ in range(args.tol_steps):
                t1 = time.perf_counter()
                ctx.step(1)
                ctx.synchronize()
                t_el += time.perf_counter() - t1
                s2 = ctx.stats()
                its.append(s2.iterations)
                errs.append(s2.max_density_error)
            cmp["plain"] = dict(iters_per_substep=float(np.mean(its)),
                                max_density_error=float(np.max(errs)),
                                ms_per_substep=1e3 * t_el / args.tol_steps,
                                particle_updates_per_s=n * args.tol_steps / t_el)
        pl, wm = cmp["plain"], cmp["warm"]
        out["jacobi"] = {"tolerance": 1e-3, "cap": 10, "substeps": args.tol_steps,
                         "plain_iters_per_substep": pl["iters_per_substep"],
                         "plain_max_density_error": pl["max_density_error"],
                         "plain_mean_final_error": pl.get("mean_final_error"),
                         "plain_error_after_iterations": pl.get("error_after_iterations"),
                         "plain_particle_updates_per_s": pl["particle_updates_per_s"],
                         "warm_iters_per_substep": wm["iters_per_substep"] if wm else None,
                         "warm_max_density_error": wm["max_density_error"] if wm else None,
                         "warm_mean_final_error": wm["mean_final_error"] if wm else None,
                         "warm_error_after_iterations":
                             wm["error_after_iterations"] if wm else None,
                         "warm_fallbacks": wm["fallbacks"] if wm else None,
                         "warm_particle_updates_per_s":
                             wm["particle_updates_per_s"] if wm else None,
                         "warm_speedup": (wm["particle_updates_per_s"] /
                                          pl["particle_updates_per_s"]) if wm else None,
                         "network": os.path.relpath(args.net, ROOT) if net else None}
        pv = cmp.get("prev")
        if pv:
            out["jacobi"].update({
                "prev_scale": args.prev_scale,
                "prev_iters_per_substep": pv["iters_per_substep"],
                "prev_mean_final_error": pv["mean_final_error"],
                "prev_error_after_iterations": pv["error_after_iterations"],
                "prev_fallbacks": pv["fallbacks"],
                "prev_particle_updates_per_s": pv["particle_updates_per_s"],
                "prev_speedup": pv["particle_updates_per_s"] / pl["particle_updates_per_s"]})
        # equal accuracy: the fewest fixed iterations with which each mode
        # reaches the plain solver's error at the cap, timed from the same state
        eq = warm_train.equal_accuracy(ctx, net, pos, vel, gpu_params(sc, iters=10),
                                       args.eq_steps, cap=10, prev_scale=args.prev_scale)
        out["jacobi"]["equal_accuracy"] = {
            k: v for k, v in eq.items() if k != "curves"}
        out["jacobi"]["equal_accuracy"]["error_by_iterations"] = {
            m: [r["mean_error"] for r in c] for m, c in eq["curves"].items()}
        ctx.upload(pos, vel)
        out["kinetic_energy_J"] = ctx.kinetic_energy()
        # the same throughput over later windows of the run: the mean neighbour
        # count and the longest lists grow as the columns collapse
        ctx.set_params(gpu_params(sc))
        out["later_windows"] = [later_window(ctx, (start_at, start), a, 20, not args.no_graph)
                                for a in (50, 100)]
    ctx.close()
    if not args.no_extras:
        # the batched-scene workload, summarised (full line: --workload batch)
        b = run_batch(args.scenes, args.batch_steps, args.warmup, graph=not args.no_graph,
                      autotune=not args.no_autotune, net_path=args.batch_net)
        out["batch"] = {k: b[k] for k in ("value", "unit", "ms_per_step", "steps",
                                          "scene_max_density_error_plain", "warm_start",
                                          "roofline")}
        # launch gaps and tails: the graph-replayed substep against the sum of
        # its kernels' durations (event-timed eager launches of the same substeps)
        ksum = b["kernels_ms_per_substep_eager"]["_sum"]
        out["batch"]["kernel_sum_ms_per_substep"] = ksum
        out["batch"]["idle_fraction"] = max(0.0, 1.0 - ksum / b["ms_per_step"])
        out["batch"]["workload"] = b["config"]["workload"]
        out["batch"]["particles"] = b["config"]["particles"]
        out["batch"]["scenes"] = b["config"]["scenes"]
    if not args.no_cpu and not args.no_extras:
        threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
        out["cpu_baseline"] = cpu_baseline(sc, args.cpu_steps, threads)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
