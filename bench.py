#!/usr/bin/env python3
"""Throughput of the DVM source iteration on one MI355X.

Workload (the configuration the headline metric is quoted on): a 200^3 image
of randomly placed overlapping solid spheres (centres uniform in the box,
radii uniform in [4, 10] voxels, added until the porosity is 0.40, PCG64 seed
2024), 4 fluid layers at inlet and outlet (208 x 200 x 200 domain), 8^3
half-range Gauss-Hermite velocities, Kn = 1, pressure drop 1 along x, diffuse
walls (accom = 1), second-order wall extrapolation.

One step = one source iteration (eight octant sweeps, wall and inlet/outlet
conditions, symmetry planes, moments) over the whole image with f resident
in HBM.  value = cell*velocity updates per second = Nfluid * 512 * steps /
wall time of the timed steps.  roofline: the sweep kernels' algorithmic HBM
bytes (16 B per update in FP64: read the previous f, write the new one)
divided by their device time from HIP events, against 8 TB/s.
cpu_baseline: the reference program itself (built from its own sources into
oracle/_ref), 2 iterations of the same workload on the host cores.

    python bench.py [--steps K] [--warmup W] [--precision fp64]
"""
import argparse
import hashlib
import json
import os
import re
import subprocess
import sys
import tempfile
import time

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

METRIC = "cell·velocity updates/s; batched solves/s + p99 latency at 1e-8 perm error"
HBM_PEAK_GBS = 8000.0
SEED = 2024


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def workload():
    from piks3d_amd import images
    from piks3d_amd.params import Params
    img = images.sphere_pack(200, 0.40, 4.0, 10.0, seed=SEED)
    p = Params(image_file_name="spheres200.raw", nx=200, ny=200, nz=200, fluid_layer=4,
               wall_ext_order=2, ref_l=1.0, nc_fundamental=4, half_range=True,
               chk_converge_step=10, max_step=2, eps=0.0, kn=1.0, press_drop=1.0, accom=1.0)
    return p, img


def cpu_baseline(p, img, nfluid, nc, threads, iters=2):
    """Time the reference program (oracle/_ref/piks3d) on `iters` iterations."""
    from piks3d_amd.params import format_para
    from piks3d_amd import images
    exe = os.path.join(HERE, "oracle", "_ref", "piks3d")
    if not os.path.exists(exe):
        return None
    with tempfile.TemporaryDirectory(prefix="piks_ref_") as d:
        images.write_raw(os.path.join(d, p.image_file_name), img)
        q = dict(p.__dict__)
        from piks3d_amd.params import Params
        pr = Params(**q)
        pr.max_step = iters
        pr.chk_converge_step = 1000
        pr.save_last = False
        pr.save_step = 1 << 30
        with open(os.path.join(d, "para.in"), "w") as fh:
            fh.write(format_para(pr))
        env = dict(os.environ, OMP_NUM_THREADS=str(threads))
        log("cpu baseline: reference program, %d threads, %d iterations" % (threads, iters))
        r = subprocess.run([exe], cwd=d, env=env, capture_output=True, text=True, timeout=900)
        m = re.search(r"Walltime=\s*([0-9.Ee+-]+)", r.stdout)
        if r.returncode != 0 or not m:
            log("reference run failed:", r.stdout[-500:], r.stderr[-500:])
            return None
        wall = float(m.group(1))
    return {"value": nfluid * nc * iters / wall, "unit": "updates/s", "cores": threads,
            "kind": "reference",
            "sample": "%d iterations of the same 208x200x200 workload, reference PIKS3D "
                      "(flang -O2 -fopenmp, 1 MPI rank), loop wall time %.3g s" % (iters, wall)}


def physical_cores():
    """Physical cores this process may run on: distinct (package, core) pairs
    of /proc/cpuinfo among the CPUs of the affinity mask (the logical count
    when the file gives no topology)."""
    try:
        allowed = os.sched_getaffinity(0)
    except AttributeError:
        allowed = set(range(os.cpu_count() or 1))
    cores, cpu, pkg = set(), None, None
    try:
        with open("/proc/cpuinfo") as fh:
            for line in fh:
                k, _, v = line.partition(":")
                k, v = k.strip(), v.strip()
                if k == "processor":
                    cpu, pkg = int(v), None
                elif k == "physical id":
                    pkg = v
                elif k == "core id" and cpu in allowed:
                    cores.add((pkg, v))
    except OSError:
        pass
    return len(cores) if cores else len(allowed)


def refined_measurement(p, img, steps, warmup, block, k64, fp64_ms_per_step):
    """The FP64 defect correction on the same workload: `warmup` plain FP64
    iterations, then `steps` iterations in blocks of `block` (one FP64
    residual iteration, block - 1 FP32 correction iterations).  Returns the
    whole-iteration rate of the timed steps, the correction sweep's roofline
    at its algorithmic 12 B per update (read the correction and the residual,
    write the correction) and K against the plain FP64 run at equal
    iteration counts.  The blocks are forced from the start of the solve,
    where a block's correction is as large as the state itself, so this K
    difference shows FP32 rounding of the whole state (about 1e-7); the
    library's own block policy stays in FP64 until the check's error is below
    1e-2 and is held to 1e-8 in K by the tests."""
    from piks3d_amd import Solver
    os.environ["PIKS_DC_BLOCK"] = "1"
    with Solver(p, img, precision="fp32") as s:
        nf, nc = s.info.nfluid, s.info.nc8 * 8
        rows = s.sweep_kind() == "rows"
        s.iterate(warmup)
        s.chk_converge()
        os.environ.pop("PIKS_DC_BLOCK")
        # the block length from here on (the library's policy would pick it
        # from the check; fixed here so that the measurement is repeatable)
        s.set_correction_block(block)
        t0 = time.perf_counter()
        s.iterate(steps)
        t1 = time.perf_counter()
        ms = s.timing()
        m, k, err = s.chk_converge()
        # correction iterations alone: the block's iterations 2..block, each
        # timed by the wall clock around the synchronous piks_iterate (the
        # whole iteration, defect-correction passes included) and its sweep
        # by HIP events
        corr = []
        for q in range(block):
            t0c = time.perf_counter()
            s.iterate(1)
            wall = (time.perf_counter() - t0c) * 1e3
            corr.append((wall, s.timing()[0]))
        n32 = s.get_info().steps_fp32
    corr = sorted(corr)[:-1]  # drop the block's FP64 iteration (the slowest)
    sweep_ms = sum(t[1] for t in corr) / len(corr)
    it_ms = sum(t[0] for t in corr) / len(corr)
    upd = nf * nc
    ach = upd * 12 / (sweep_ms / 1e3) / 1e9
    dt = t1 - t0
    return {
        "block": block, "value": upd * steps / dt, "unit": "updates/s", "ms_per_step": dt / steps * 1e3,
        "speedup_vs_fp64": fp64_ms_per_step / (dt / steps * 1e3),
        "correction_iteration_ms": round(it_ms, 4), "correction_sweep_ms": round(sweep_ms, 4),
        "correction_roofline": {"bound": "hbm", "achieved": round(ach, 1), "peak": HBM_PEAK_GBS,
                                "unit": "GB/s", "frac": round(ach / HBM_PEAK_GBS, 4), "bytes_per_update": 12,
                                "kernel": "k_sweep_pencil<float, 2, false>" if rows else "k_sweep1<float, false, 2>"},
        "k_rel_diff_vs_fp64_blocks_from_rest": abs(k - k64) / abs(k64) if k64 else abs(k - k64),
        "steps_compared": warmup + steps,
        "fp32_iterations": int(n32)}


def traffic_from_profiles(workload_name):
    path = os.path.join(HERE, "profiles", "traffic_%s.json" % workload_name)
    if os.path.exists(path):
        with open(path) as fh:
            return json.load(fh).get("bytes_per_step")
    return None


SERVE_SIDES = (32, 48, 64, 96, 128)


def serve_specs(nreq, seed, max_step, eps):
    """The serving stream's requests without their images: nreq seeded
    sphere packs, side uniform over SERVE_SIDES, porosity U[0.3, 0.5], Kn
    log-uniform over [0.01, 10], velocity grid 6^3 for Kn < 0.1, 8^3 for
    Kn < 1, else 12^3 (half-range), 4 fluid layers, unit pressure drop.
    Returns (Params, porosity, image seed) per request."""
    import numpy as np
    from piks3d_amd.params import Params
    rng = np.random.Generator(np.random.PCG64(seed))
    specs = []
    for q in range(nreq):
        side = int(rng.choice(SERVE_SIDES))
        phi = float(rng.uniform(0.3, 0.5))
        kn = float(10.0 ** rng.uniform(-2.0, 1.0))
        nc = 3 if kn < 0.1 else (4 if kn < 1.0 else 6)
        p = Params(nx=side, ny=side, nz=side, fluid_layer=4, wall_ext_order=2, nc_fundamental=nc,
                   half_range=True, exact_quadrature=(nc == 3), chk_converge_step=10,
                   max_step=max_step, eps=eps, kn=kn, press_drop=1.0, accom=1.0)
        specs.append((p, phi, seed * 100003 + q))
    return specs


def serve_image(p, phi, img_seed):
    from piks3d_amd import images
    return images.sphere_pack(p.nx, phi, 4.0, 10.0, seed=img_seed)


def serve_workload(nreq, seed, max_step, eps):
    """The serving stream (serve_specs) with images and update counts."""
    from piks3d_amd import preprocess
    reqs = []
    for q, (p, phi, img_seed) in enumerate(serve_specs(nreq, seed, max_step, eps)):
        img = serve_image(p, phi, img_seed)
        _, info = preprocess(p, img)
        reqs.append((p, img, info.nfluid * 8 * p.nc_fundamental ** 3))
        if (q + 1) % 16 == 0:
            log("generated %d of %d" % (q + 1, nreq))
    return reqs


def serve_bench(args):
    """Poisson arrivals into the request server; one JSON line."""
    import numpy as np
    from piks3d_amd import REQ_DONE, Server
    log("generating %d requests" % args.requests)
    reqs = serve_workload(args.requests, args.seed, args.max_step, args.eps)
    rng = np.random.Generator(np.random.PCG64(args.seed + 1))
    arrivals = np.cumsum(rng.exponential(1.0 / args.rate, len(reqs)))
    with Server(max_slots=args.slots, prep_threads=args.prep_threads) as srv:
        t0 = time.perf_counter()
        tickets = []
        for (p, img, _), at in zip(reqs, arrivals):
            delay = t0 + at - time.perf_counter()
            if delay > 0:
                time.sleep(delay)
            tickets.append(srv.submit(p, img, precision=args.precision))
            if len(tickets) % 32 == 0:
                log("%d submitted, %.1f s" % (len(tickets), time.perf_counter() - t0))
        log("all %d submitted after %.1f s" % (len(tickets), time.perf_counter() - t0))
        res = []
        for q, t in enumerate(tickets):
            res.append(srv.wait(t))
            if (q + 1) % 8 == 0:
                log("%d done, %.1f s" % (q + 1, time.perf_counter() - t0))
        wall = time.perf_counter() - t0
    ok = [r for r in res if r["status"] == REQ_DONE]
    lat = np.array([r["total_ms"] for r in ok])
    updates = sum(u * r["steps"] for (_, _, u), r in zip(reqs, res) if r["status"] == REQ_DONE)
    out = {
        "metric": "batched solves/s + p99 latency (serving stream)", "value": len(ok) / wall,
        "unit": "solves/s", "higher_is_better": True, "n_gpus": 1,
        "p50_ms": float(np.percentile(lat, 50)), "p99_ms": float(np.percentile(lat, 99)),
        "mean_run_ms": float(np.mean([r["run_ms"] for r in ok])),
        "updates_per_s": updates / wall, "wall_s": wall, "failed": len(res) - len(ok),
        "converged": int(sum(r["converged"] for r in ok)),
        "dtype": "f64" if args.precision == "fp64" else "f32+f64", "data": "synthetic",
        "config": {"workload": "serving_stream_%d" % args.requests, "sides": list(SERVE_SIDES),
                   "porosity": [0.3, 0.5], "kn": [0.01, 10], "arrival_rate_per_s": args.rate,
                   "slots": args.slots, "max_step": args.max_step, "eps": args.eps,
                   "precision": args.precision, "seed": args.seed},
    }
    print(json.dumps(out))


def kn_sweep_bench(args):
    """Multi-RHS Knudsen sweep: one 160^3 Gaussian-random-field image
    (correlation length 5 voxels, porosity 0.25, percolating in x), 32 Kn
    log-spaced over [1e-3, 10], 8^3 velocities, solved as groups of right-hand
    sides sharing the geometry (one sweep launch per iteration for a group),
    in --precision (fp32: the FP64 defect correction with FP32 correction
    iterations); a few Kn are re-solved in plain FP64 for the same number of
    iterations and compared."""
    import numpy as np
    from piks3d_amd import MultiSolver, images
    from piks3d_amd.params import Params
    img = images.gaussian_field(160, 0.25, 5.0, seed=args.seed)
    p = Params(nx=160, ny=160, nz=160, fluid_layer=4, wall_ext_order=2, nc_fundamental=4, half_range=True,
               chk_converge_step=10, max_step=args.max_step, eps=args.eps, kn=1.0, press_drop=1.0, accom=1.0)
    kns = np.logspace(-3, 1, args.nkn)
    perm, steps, conv = np.zeros(len(kns)), np.zeros(len(kns), int), np.zeros(len(kns), bool)
    updates, wall, solve_wall = 0.0, 0.0, 0.0
    for g0 in range(0, len(kns), args.group):
        ks = list(kns[g0:g0 + args.group])
        t = time.perf_counter()
        with MultiSolver(p, img, ks, precision=args.precision) as ms:
            nf = ms.info.nfluid
            ts = time.perf_counter()
            r = ms.solve()
            solve_wall += time.perf_counter() - ts
        dt = time.perf_counter() - t
        wall += dt
        updates += nf * 512 * r["steps"] * len(ks)
        perm[g0:g0 + len(ks)] = r["permeability"]
        steps[g0:g0 + len(ks)] = r["steps"]
        conv[g0:g0 + len(ks)] = np.asarray(r["error"]) <= args.eps
        log("Kn %.3g..%.3g: %d steps (%d FP32), %.1f s" % (ks[0], ks[-1], r["steps"], r["steps32"], dt))
    # every Kn against the plain FP64 solve of the same length: FP64
    # several-Kn contexts over the same groups (each right-hand side of one
    # equals its single solve bit for bit); an FP64 sweep checks itself
    check = list(range(len(kns))) if args.precision != "fp64" else [0, len(kns) - 1]
    rel = [0.0] * len(kns)
    t64 = time.perf_counter()
    for g0 in range(0, len(kns), args.group):
        qs = [q for q in range(g0, min(g0 + args.group, len(kns))) if q in check]
        if not qs:
            continue
        with MultiSolver(p, img, [kns[q] for q in qs], precision="fp64") as ms:
            r64 = ms.solve(max_step=int(steps[qs[0]]), eps=0.0)
        for q, k64 in zip(qs, r64["permeability"]):
            rel[q] = abs(perm[q] - k64) / abs(k64)
    log("FP64 check of %d Kn: %.1f s, largest relative K difference %.3e" % (
        len(check), time.perf_counter() - t64, max(rel[q] for q in check)))
    rel = [rel[q] for q in check]
    out = {
        "metric": "multi-RHS Knudsen sweep: cell*velocity updates/s", "value": updates / wall,
        "unit": "updates/s", "higher_is_better": True, "n_gpus": 1, "wall_s": wall,
        "solve_updates_per_s": updates / solve_wall, "solve_wall_s": solve_wall,
        "dtype": "f64" if args.precision == "fp64" else "f32+f64", "data": "synthetic",
        "kn": [float(k) for k in kns], "permeability": [float(k) for k in perm],
        "steps": [int(x) for x in steps], "converged": [bool(x) for x in conv],
        "check_vs_fp64": {"kn": [float(kns[q]) for q in check], "rel_diff": rel, "max_rel_diff": max(rel)},
        "config": {"workload": "grf160_phi025_l5_kn32", "group": args.group, "max_step": args.max_step,
                   "eps": args.eps, "precision": args.precision, "seed": args.seed},
    }
    print(json.dumps(out))


def large_bench(args):
    """The large single solve: a 300^3 Gaussian-random-field image
    (correlation length 6, porosity 0.20, percolating in x), 8^3 velocities,
    Kn in {0.01, 1, 10}: plain FP64 iterations and the defect correction in
    blocks of --dc-block (refined_measurement), throughput over a few
    iterations each."""
    from piks3d_amd import Solver, images
    from piks3d_amd.params import Params
    img = images.gaussian_field(300, 0.20, 6.0, seed=args.seed)
    rows = []
    for kn in (0.01, 1.0, 10.0):
        p = Params(nx=300, ny=300, nz=300, fluid_layer=4, wall_ext_order=2, nc_fundamental=4, half_range=True,
                   chk_converge_step=10, max_step=2, kn=kn, press_drop=1.0, accom=1.0)
        with Solver(p, img, precision="fp64") as s:
            s.iterate(args.warmup)
            t = time.perf_counter()
            s.iterate(args.steps)
            dt = time.perf_counter() - t
            ms = s.timing()
            k64 = s.chk_converge()[1]
            upd = s.info.nfluid * 512 * args.steps
            rows.append({"kn": kn, "precision": "fp64", "updates_per_s": upd / dt,
                         "sweep_ms_per_step": ms[0] / args.steps, "ms_per_step": dt / args.steps * 1e3,
                         "device_gb": s.info.device_bytes / 1e9, "fluid_cells": s.info.nfluid})
            log("Kn %g fp64: %.3g updates/s, %.1f ms/step, %.1f GB" % (kn, upd / dt, dt / args.steps * 1e3,
                                                                       s.info.device_bytes / 1e9))
        if args.dc_block > 1:
            r = refined_measurement(p, img, args.steps, args.warmup, args.dc_block, k64, dt / args.steps * 1e3)
            rows.append({"kn": kn, "precision": "refined", "updates_per_s": r["value"],
                         "ms_per_step": r["ms_per_step"], "speedup_vs_fp64": r["speedup_vs_fp64"],
                         "correction_sweep_ms": r["correction_sweep_ms"], "block": args.dc_block})
            log("Kn %g refined (blocks of %d): %.3g updates/s (%.2fx FP64)" % (kn, args.dc_block, r["value"],
                                                                             r["speedup_vs_fp64"]))
    print(json.dumps({"metric": "large single solve: cell*velocity updates/s", "unit": "updates/s",
                      "value": min(r["updates_per_s"] for r in rows if r["precision"] == "fp64"),
                      "higher_is_better": True, "n_gpus": 1, "data": "synthetic", "rows": rows,
                      "config": {"workload": "grf300_phi020_l6", "steps": args.steps, "warmup": args.warmup,
                                 "seed": args.seed}}))


# The reference's converged permeability for the 64^3 sphere configuration
# (its own run stops at iteration 80 with K = 1.86415031246455858e-02; the
# value is also held by tests/golden/c1_sphere64.npz).
C1_K_REFERENCE = 1.86415031246455858e-02


def c1_bench(args):
    """The CPU-runnable configuration to convergence: 64^3 image with one
    centred solid sphere of radius 28, 4 fluid layers at inlet and outlet,
    8^3 half-range velocities, Kn 0.1, unit pressure drop, check every 10
    iterations, eps 1e-6.  GPU (FP64, both reduction modes) time to solution
    beside the reference program run to convergence on the host cores."""
    from piks3d_amd import Solver, images
    from piks3d_amd.params import Params, format_para
    img = images.centered_sphere(64, 28.0)
    p = Params(image_file_name="sphere64.raw", nx=64, ny=64, nz=64, fluid_layer=4, wall_ext_order=2,
               nc_fundamental=4, half_range=True, chk_converge_step=10, max_step=100000, eps=1e-6,
               kn=0.1, press_drop=1.0, accom=1.0)
    rows = {}
    for exact in (False, True):
        t = time.perf_counter()
        with Solver(p, img, precision="fp64", exact_order=exact) as s:
            t1 = time.perf_counter()
            r = s.solve()
            t2 = time.perf_counter()
            nf, nc = s.info.nfluid, s.info.nc8 * 8
        rows["exact" if exact else "fast"] = {
            "steps": r["steps"], "permeability": r["permeability"],
            "rel_diff_vs_reference": abs(r["permeability"] - C1_K_REFERENCE) / C1_K_REFERENCE,
            "setup_s": t1 - t, "solve_s": t2 - t1, "updates_per_s": nf * nc * r["steps"] / (t2 - t1)}
        log("C1 %s: %d steps, K %.17e, solve %.3f s" % ("exact" if exact else "fast", r["steps"],
                                                       r["permeability"], t2 - t1))
    cpu = None
    exe = os.path.join(HERE, "oracle", "_ref", "piks3d")
    if not args.no_cpu_baseline and os.path.exists(exe):
        with tempfile.TemporaryDirectory(prefix="piks_ref_") as d:
            images.write_raw(os.path.join(d, p.image_file_name), img)
            pr = Params(**dict(p.__dict__))
            pr.save_last = False
            pr.save_step = 1 << 30
            with open(os.path.join(d, "para.in"), "w") as fh:
                fh.write(format_para(pr))
            env = dict(os.environ, OMP_NUM_THREADS=str(args.cpu_threads))
            log("C1 reference program to convergence, %d threads" % args.cpu_threads)
            r = subprocess.run([exe], cwd=d, env=env, capture_output=True, text=True, timeout=900)
            m = re.search(r"Walltime=\s*([0-9.Ee+-]+),\s*Steps=\s*([0-9]+)", r.stdout)
            if r.returncode == 0 and m:
                wall, steps = float(m.group(1)), int(m.group(2))
                cpu = {"value": wall, "unit": "s", "cores": args.cpu_threads, "kind": "reference",
                       "steps": steps, "updates_per_s": nf * nc * steps / wall,
                       "sample": "the whole run to convergence, reference PIKS3D (flang -O2 -fopenmp, "
                                 "1 MPI rank)"}
            else:
                log("reference run failed:", r.stdout[-500:], r.stderr[-500:])
    fast = rows["fast"]
    print(json.dumps({
        "metric": "time to converged permeability, CPU-runnable configuration", "value": fast["solve_s"],
        "unit": "s", "higher_is_better": False, "n_gpus": 1, "dtype": "f64", "data": "synthetic",
        "updates_per_s": fast["updates_per_s"], "rows": rows, "cpu_baseline": cpu,
        "config": {"workload": "sphere64_r28_kn01_v8", "fluid_cells": nf, "velocities": nc,
                   "eps": p.eps, "chk_converge_step": p.chk_converge_step}}))


def flow_compare_bench(args):
    """The single-launch sweep (PIKS_SWEEP_FLOW=1, the default where it
    applies) beside the hyperplane launches (PIKS_SWEEP_FLOW=0) on sphere packs of the headline workload's kind
    (porosity 0.40, radii 4-10, seed 2024, 4 fluid layers) at the sizes of
    --flow-sizes: sweep device time per iteration (mean over --steps
    iterations after --warmup untimed ones) and whether the two paths leave the
    same state (f compared bit for bit up to 100^3, above that the moments
    and the check), in FP64."""
    import numpy as np
    from piks3d_amd import Solver, images
    from piks3d_amd.params import Params
    rows = []
    for n in [int(v) for v in args.flow_sizes.split(",")]:
        img = images.sphere_pack(n, 0.40, 4.0, 10.0, seed=SEED)
        p = Params(nx=n, ny=n, nz=n, fluid_layer=4, wall_ext_order=2, ref_l=1.0, nc_fundamental=4,
                   half_range=True, chk_converge_step=10, max_step=2, eps=0.0, kn=1.0, press_drop=1.0,
                   accom=1.0)
        res = {}
        for mode in ("hyperplanes", "single_launch"):
            os.environ["PIKS_SWEEP_FLOW"] = "1" if mode == "single_launch" else "0"
            with Solver(p, img, precision="fp64") as s:
                s.iterate(max(1, args.warmup))
                t = time.perf_counter()
                s.iterate(args.steps)
                wall = time.perf_counter() - t
                sweep_ms = s.timing()[0] / args.steps
                chk = s.chk_converge()
                state = s.f() if n <= 100 else np.stack(s.macro())
                nf = s.info.nfluid
            res[mode] = (sweep_ms, wall / args.steps * 1e3, chk, state)
            log("%d^3 %s: sweep %.3f ms/iteration, iteration %.3f ms" % (n, mode, sweep_ms,
                                                                        wall / args.steps * 1e3))
        os.environ.pop("PIKS_SWEEP_FLOW", None)
        h, f = res["hyperplanes"], res["single_launch"]
        rows.append({"n": n, "fluid_cells": nf, "sweep_ms_hyperplanes": h[0], "sweep_ms_single_launch": f[0],
                     "iteration_ms_hyperplanes": h[1], "iteration_ms_single_launch": f[1],
                     "speedup": h[0] / f[0], "same_bits": bool(h[2] == f[2] and np.array_equal(h[3], f[3])),
                     "compared": "f" if n <= 100 else "moments and check"})
    print(json.dumps({"metric": "sweep device time per iteration, single launch vs hyperplane launches",
                      "unit": "ms", "higher_is_better": False, "n_gpus": 1, "dtype": "f64", "data": "synthetic",
                      "rows": rows, "config": {"workload": "spheres_phi040_r4-10_kn1_v8", "steps": args.steps,
                                                         "warmup": max(1, args.warmup)}}))


def c2_solve_bench(args):
    """The 200^3 pack solved to the reference's criterion (check every 10
    iterations, eps = --eps, at most --max-step iterations) in plain FP64 and
    as the refined solve (the FP64 defect correction, FP32 correction
    iterations in blocks chosen from each check): iterations, the share of
    FP32 iterations, time to solution, whole-solve updates/s and the
    permeability difference.  With
    wallExtOrder 2 the reference's own iteration grows without bound on this
    pack after about a hundred iterations, so solves use --wall-order 1."""
    from piks3d_amd import Solver
    p, img = workload()
    p.chk_converge_step = 10
    p.wall_ext_order = args.wall_order
    rows, hist = {}, {}
    for prec in ("fp64", "fp32"):
        with Solver(p, img, precision=prec) as s:
            nf, nc = s.info.nfluid, s.info.nc8 * 8
            t = time.perf_counter()

            def progress(step, m, k, e):
                if step % 500 == 0:
                    log("C2 %s: step %d, K %.12e, error %.3e" % (prec, step, k, e))
            r = s.solve(max_step=args.max_step, eps=args.eps, callback=progress)
            dt = time.perf_counter() - t
        hist[prec] = {h[0]: h[2] for h in r["history"]}
        rows[prec] = {"steps": r["steps"], "steps_fp32": r.get("steps32", 0),
                      "fp32_share": r.get("steps32", 0) / max(r["steps"], 1), "permeability": r["permeability"],
                      "error": r["error"], "solve_s": dt, "updates_per_s": nf * nc * r["steps"] / dt}
        log("C2 %s: %d steps (%d FP32), K %.12e, %.2f s" % (prec, r["steps"], r.get("steps32", 0),
                                                          r["permeability"], dt))
    a, b = rows["fp64"], rows["fp32"]
    # K at every check both solves reached (equal iteration counts)
    common = sorted(set(hist["fp64"]) & set(hist["fp32"]))
    kdiff = max((abs(hist["fp32"][q] - hist["fp64"][q]) / abs(hist["fp64"][q]) for q in common
                 if hist["fp64"][q]), default=None)
    print(json.dumps({
        "metric": "time to solution, 200^3 sphere pack, plain FP64 vs refined", "value": b["solve_s"],
        "unit": "s", "higher_is_better": False, "n_gpus": 1, "data": "synthetic", "rows": rows,
        "speedup_refined_vs_fp64": a["solve_s"] / b["solve_s"],
        "rel_diff_permeability": abs(a["permeability"] - b["permeability"]) / abs(a["permeability"]),
        "max_rel_diff_permeability_at_equal_checks": kdiff, "checks_compared": len(common),
        "config": {"workload": "spheres200_phi040_kn1_v8", "eps": args.eps, "max_step": args.max_step,
                   "chk_converge_step": 10, "wall_ext_order": args.wall_order}}))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--precision", default="fp64", choices=["fp64", "fp32"])
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-threads", type=int, default=0,
                    help="host threads of the CPU baseline (0: every physical core of the affinity mask)")
    ap.add_argument("--dc-block", type=int, default=20,
                    help="block length of the defect-correction measurement in the bench line")
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="MIB",
                    help="only run a device-to-device copy of MIB MiB three times (for scaling "
                         "FETCH_SIZE / WRITE_SIZE counters) and exit")
    ap.add_argument("--serve", action="store_true",
                    help="run the serving stream instead (Poisson arrivals into the request server)")
    ap.add_argument("--kn-sweep", action="store_true",
                    help="run the multi-RHS Knudsen sweep on a 160^3 random field instead")
    ap.add_argument("--c2-solve", action="store_true",
                    help="the 200^3 pack to convergence, plain FP64 and refined")
    ap.add_argument("--wall-order", type=int, default=2,
                    help="--c2-solve: wallExtOrder (the reference's iteration diverges on this pack with 2)")
    ap.add_argument("--c1", action="store_true",
                    help="the 64^3 sphere configuration to convergence, GPU and reference program")
    ap.add_argument("--flow-compare", action="store_true",
                    help="single-launch sweep beside the hyperplane launches at --flow-sizes")
    ap.add_argument("--flow-sizes", default="40,64,100,200")
    ap.add_argument("--large", action="store_true",
                    help="run the 300^3 random-field single solve at Kn 0.01, 1, 10 instead")
    ap.add_argument("--nkn", type=int, default=32)
    ap.add_argument("--group", type=int, default=16)
    ap.add_argument("--requests", type=int, default=256)
    ap.add_argument("--rate", type=float, default=8.0, help="serving: mean arrivals per second")
    ap.add_argument("--slots", type=int, default=8)
    ap.add_argument("--prep-threads", type=int, default=8)
    ap.add_argument("--max-step", type=int, default=400)
    ap.add_argument("--eps", type=float, default=1e-6)
    ap.add_argument("--seed", type=int, default=7)
    args = ap.parse_args()
    if args.cpu_threads <= 0:
        args.cpu_threads = physical_cores()
    if args.gpus != 1:
        print("bench.py measures one GPU only: the library has no multi-GPU path "
              "(run with --gpus 1)", file=sys.stderr)
        sys.exit(2)
    if args.copy_calibration:
        import torch
        n = args.copy_calibration << 20
        src = torch.ones(n, dtype=torch.uint8, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        log("copied %d bytes three times" % n)
        return
    if args.serve:
        serve_bench(args)
        return
    if args.kn_sweep:
        kn_sweep_bench(args)
        return
    if args.large:
        large_bench(args)
        return
    if args.c1:
        c1_bench(args)
        return
    if args.flow_compare:
        flow_compare_bench(args)
        return
    if args.c2_solve:
        c2_solve_bench(args)
        return

    try:
        import torch
        sync = torch.cuda.synchronize if torch.cuda.is_available() else (lambda: None)
    except Exception:  # torch is plumbing only; piks_iterate synchronizes its stream itself
        sync = lambda: None  # noqa: E731

    from piks3d_amd import Solver
    if args.precision != "fp64":
        sys.exit("bench.py: the benchmark line runs plain FP64 iterations and reports the refined precision "
                 "(the defect correction) in its 'refined' object; --precision applies to --serve and --kn-sweep")
    log("generating the 200^3 sphere pack")
    p, img = workload()
    t = time.perf_counter()
    s = Solver(p, img, precision="fp64")
    info = s.info
    log("set-up %.1f s: Nfluid %d, walls %d, corners %d, device memory %.1f GB" % (
        time.perf_counter() - t, info.nfluid, info.nwall, info.ncorner, info.device_bytes / 1e9))
    nc = info.nc8 * 8
    flow = s.sweep_kind() == "rows"
    log("sweep: %s" % ("one launch per iteration (k_sweep_pencil)" if flow else "one launch per hyperplane"))
    if args.warmup:
        s.iterate(args.warmup)
    log("warm-up done (%d steps)" % args.warmup)
    sync()
    t0 = time.perf_counter()
    s.iterate(args.steps)
    sync()
    t1 = time.perf_counter()
    ms = s.timing()
    elapsed = t1 - t0
    updates = info.nfluid * nc * args.steps
    value = updates / elapsed
    bytes_per_update = 16
    sweep_s = ms[0] / 1e3
    achieved = updates * bytes_per_update / sweep_s / 1e9
    m, k, err = s.chk_converge()
    log("timed %d steps in %.3f s: %.4g updates/s; phases (ms/step): sweep %.3f, walls+bc %.3f, "
        "moments %.3f; K after %d steps = %.6e" % (
            args.steps, elapsed, value, ms[0] / args.steps, ms[1] / args.steps, ms[2] / args.steps,
            args.warmup + args.steps, k))
    s.close()
    refined = None
    if args.dc_block > 1:
        refined = refined_measurement(p, img, args.steps, args.warmup, args.dc_block, k,
                                      elapsed / args.steps * 1e3)
        log("defect correction, blocks of %d: %.4g updates/s (%.2fx FP64), correction iteration %.3f ms "
            "(sweep %.3f ms, %.1f %% of HBM at 12 B/update), K rel diff %.2e (blocks from rest)" % (
                args.dc_block, refined["value"], refined["speedup_vs_fp64"], refined["correction_iteration_ms"],
                refined["correction_sweep_ms"], 100 * refined["correction_roofline"]["frac"],
                refined["k_rel_diff_vs_fp64_blocks_from_rest"]))

    wl = "spheres200_phi040_kn1_v8"
    roof = {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBS, 4),
            "traffic": traffic_from_profiles(wl + ("_rows" if flow else "")),
            "kernel": "k_sweep_pencil" if flow else "k_sweep1<double, false>",
            "bytes_per_update": bytes_per_update,
            "sweep_ms_per_step": round(ms[0] / args.steps, 4)}
    cpu = None
    if not args.no_cpu_baseline:
        cpu = cpu_baseline(p, img, info.nfluid, nc, args.cpu_threads)
    out = {
        "metric": METRIC, "value": value, "unit": "updates/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": elapsed / args.steps * 1e3,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": wl, "image": "200^3 overlapping spheres r~U[4,10], porosity 0.40, seed %d" % SEED,
                   "image_sha256": hashlib.sha256(img.tobytes()).hexdigest(),
                   "domain": [info.nx, info.ny, info.nz], "fluid_cells": info.nfluid,
                   "velocities": nc, "kn": p.kn, "precision": "fp64"},
        "roofline": roof,
        "whole_iteration_roofline": {"achieved": round(updates * bytes_per_update / elapsed / 1e9, 1),
                                     "frac": round(updates * bytes_per_update / elapsed / 1e9 / HBM_PEAK_GBS, 4)},
        "refined": refined,
        "cpu_baseline": cpu,
        "phase_ms_per_step": [round(x / args.steps, 4) for x in ms[:3]],
    }
    print(json.dumps(out))


if __name__ == "__main__":
    main()
