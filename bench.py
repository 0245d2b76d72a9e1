#!/usr/bin/env python3
"""Gradient throughput of the constant-density acoustic FWI path on one MI355X.

Workload (the 2D layered case): 1001 x 301 nodes at dx = 10 m (1041 x 341
padded with 20 PML cells per side), velocities 1500-4500 m/s in 12 seeded
dipping layers times a smoothed (150 m) 5 % random field, 16 Ricker sources
(8 Hz) at 20 m depth, 1001 receivers at 20 m, nt = 3000 at the CFL step,
FP32, spatial order 8.  One "step" is one full misfit gradient of all 16
shots: forward propagation recording traces and keeping dWaveOp, the misfit
0.5*dt*||d - d_obs||^2, and the adjoint propagation with the FP64 imaging
condition and the PML fold, through the torch.autograd.Function wrapper.

value  = 2 * sum_shots(N_pad * nt) / seconds per gradient  (Gpt-updates/s),
         recompute steps of a checkpoint schedule are not counted.
checkpointed = the same batched gradient under an 8 GiB memory budget: the
         forward keeps checkpoints, the adjoint recomputes each segment's
         dWaveOp; its gradient equals the store-all one bit for bit.
plain  = the same gradient with one shot per launch (16 shot loops).
c4_3d  = the 3D checkpointed gradient (--workload c4: 8 shots of 288^3,
         nt 2000, FP32 order 8), one timed gradient in a child process.
roofline: the adjoint kernel (the dominant one): algorithmic bytes per
         launch (FP32 fields: u_k, u_k-1, C read, u_k+1 written = 16 B per
         node; imaging: dWaveOp read 4 B + FP64 accumulator read/write 16 B;
         PML nodes +16 B for Phix, Phiz read/write) over its average launch
         time from HIP events on the launch stream, against 8 TB/s.
cpu_baseline: PySIT's own step kernel (cda_time_scalar_2D<float, 8>,
         compiled here from the reference sources with the reference's flags
         into oracle/_ref) stepping the same padded grid on the host cores,
         one shot per thread; falls back to the oracle restatement.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)

HBM_PEAK_GBS = 8000.0
METRIC = "fwd+adjoint gradient Gpt-updates/s, % HBM roofline: batched-ckpt vs plain"


def parse():
    p = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=3)
    p.add_argument("--warmup", type=int, default=1)
    p.add_argument("--shots", type=int, default=16)
    p.add_argument("--nt", type=int, default=3000)
    p.add_argument("--no-plain", action="store_true", help="skip the one-shot-per-launch comparison")
    p.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    p.add_argument("--no-accuracy", action="store_true", help="skip the FP64 comparison gradient")
    p.add_argument("--no-3d", action="store_true",
                   help="c2: skip the 3D checkpointed gradient run in a child process after the 2D legs")
    p.add_argument("--cpu-seconds", type=float, default=6.0, help="target seconds per CPU baseline leg")
    p.add_argument("--tile-x", type=int, default=None)
    p.add_argument("--memory-budget-gb", type=float, default=None)
    p.add_argument("--ckpt-budget-gb", type=float, default=8.0,
                   help="c2: memory budget of the checkpointed gradient leg (0: skip it)")
    p.add_argument("--profile-run", action="store_true", help="minimal run for rocprofv3 (no plain, no CPU)")
    p.add_argument("--workload", choices=["c1", "c2", "c3", "c4", "c5"], default="c2",
                   help="c2: the headline 16-shot gradient; c3: 64 shots of uneven aperture and length; "
                        "c4: the 3D 256^3 8-shot checkpointed gradient (use --steps 1 --warmup 0); "
                        "c5: the multi-band LBFGS FWI loop (FP32, then FP64 for comparison)")
    p.add_argument("--write-traffic", nargs=2, metavar=("FETCH_CSV", "WRITE_CSV"),
                   help="write the traffic summary under profiles/ from the counter files of the two --pmc-run "
                        "profiles (FETCH_SIZE, WRITE_SIZE) and exit (no GPU needed)")
    p.add_argument("--fwi-iterations", type=int, default=20, help="c5: LBFGS iterations per band")
    p.add_argument("--fwi-bands", default="3,5,8", help="c5: Ricker peak frequencies (Hz), low to high")
    p.add_argument("--pmc-run", action="store_true",
                   help="short run for rocprofv3 --pmc: a 256 MiB elementwise calibration kernel, then one "
                        "gradient of the workload over --nt slots (default 40)")
    return p.parse_args()


def algorithmic_bytes(shapes_and_pml, itemsize, dim=2):
    """Algorithmic HBM bytes of one launch over all shots, the path's byte
    model (s = itemsize, per padded node per time step):

    forward: read u_k, u_{k-1} and the coefficient, write u_{k+1} (4s);
    adjoint: the same (4s) plus the imaging condition, one stored forward
    quantity read (s) and the FP64 accumulator read and written (16).  PML
    nodes add Phix and Phiz read and written (4s) in either direction, in 3D
    Phix, Phiy, Phiz and psi (8s).  For FP32 this is 26 + 16 f_pml bytes per
    gradient grid-point update in 2D, 26 + 32 f_pml in 3D."""
    fwd = adj = 0.0
    for npts, npml in shapes_and_pml:
        base = 4 * itemsize * npts
        pml = (4 if dim == 2 else 8) * itemsize * npml
        fwd += base + pml
        adj += base + pml + (itemsize + 16) * npts
    return fwd, adj


def pml_nodes(shape, pads):
    inner = 1
    for n, (l, r) in zip(shape, pads):
        inner *= n - l - r
    return int(np.prod(shape)) - inner


def cpu_baseline(shape, pml_pairs, dt, deltas, seconds):
    """Reference step kernel timed on the host cores, one shot per thread."""
    from concurrent.futures import ThreadPoolExecutor
    from oracle import oracle as O
    kind = "reference" if O.ref_available(fast=True) else "port"
    use_ref = kind == "reference"
    nx, nz = shape
    n = nx * nz
    rng = np.random.default_rng(0)
    (xl, xr), (zl, zr) = pml_pairs

    def run(nsteps):
        f = [rng.standard_normal(n).astype(np.float32) * 1e-3 for _ in range(6)]
        f[4] = np.full(n, 3000.0, np.float32)
        t0 = time.perf_counter()
        for _ in range(nsteps):
            px, pz, up = O.step2d(8, f[0], f[1], f[2], f[3], f[4], f[5], xl, xr, zl, zr, dt, deltas[0],
                                  deltas[1], nx, nz, dtype=np.float32, use_ref=use_ref, fast=True)
            f[0], f[3], f[1], f[2] = f[3], up, px, pz
        return time.perf_counter() - t0

    t_probe = run(3) / 3
    steps = max(3, int(seconds / max(t_probe, 1e-6)))
    t1 = run(steps)
    single = n * steps / t1 / 1e9
    threads = min(len(os.sched_getaffinity(0)), 16)
    with ThreadPoolExecutor(threads) as ex:
        t0 = time.perf_counter()
        list(ex.map(run, [steps] * threads))
        tm = time.perf_counter() - t0
    multi = n * steps * threads / tm / 1e9
    # the reference's OpenMP variants (orders 4 and 6 only), one shot over all threads
    omp = {}
    if use_ref:
        os.environ.setdefault("OMP_NUM_THREADS", str(threads))
        for order in (4, 6):
            f = [rng.standard_normal(n).astype(np.float32) * 1e-3 for _ in range(6)]
            f[4] = np.full(n, 3000.0, np.float32)

            def omp_steps(k):
                t0 = time.perf_counter()
                for _ in range(k):
                    px, pz, up = O.step2d(order, f[0], f[1], f[2], f[3], f[4], f[5], xl, xr, zl, zr, dt,
                                          deltas[0], deltas[1], nx, nz, dtype=np.float32, use_ref=True,
                                          fast=True, omp=True)
                    f[0], f[3], f[1], f[2] = f[3], up, px, pz
                return time.perf_counter() - t0
            tp = omp_steps(3) / 3
            k = max(3, int(0.5 * seconds / max(tp, 1e-6)))
            omp[f"order{order}"] = n * k / omp_steps(k) / 1e9
        omp["threads"] = int(os.environ["OMP_NUM_THREADS"])
    cpu = "unknown"
    try:
        with open("/proc/cpuinfo") as fh:
            cpu = next(l.split(":", 1)[1].strip() for l in fh if l.startswith("model name"))
    except (OSError, StopIteration):
        pass
    return {"value": multi, "unit": "Gpt-updates/s", "cores": threads, "kind": kind,
            "single_thread": single,
            "openmp_variant": omp or None,
            "host": {"nproc": os.cpu_count(), "affinity": len(os.sched_getaffinity(0)), "cpu": cpu},
            "sample": (f"{steps} steps of cda_time_scalar_2D<float,8> on the {nx}x{nz} padded grid per thread, "
                       f"{threads} threads (one shot each), -O3 -fopenmp -ffast-math; "
                       f"single thread {single:.4f} Gpt/s; the step-kernel rate bounds the CPU gradient rate "
                       f"from above (imaging and dWaveOp work not counted); openmp_variant: the reference's "
                       f"OpenMP step kernels of orders 4 and 6 (2D_4.h, 2D_6.h) on one shot over all threads")}


def cpu_gradient(solver, shot, seconds):
    """One shot's FP64 gradient on the host: the oracle's loops (its C
    restatement of the reference's step and of forward_model / migrate_shot)
    built with the reference's flags (-O3 -fopenmp -ffast-math), node loops
    over all host threads.  The oracle's migrate replays the forward pass to
    regenerate dWaveOp, so one gradient is four propagations (residual
    forward, checkpoint pass, dWaveOp recompute, adjoint); the rate counts the
    metric's two.  The full step count when it fits ``seconds``, else the
    first steps of the shot (stated in ``sample``)."""
    from tests.problems import oracle_from_solver
    from oracle import oracle as O
    threads = min(len(os.sched_getaffinity(0)), 16)
    os.environ.setdefault("OMP_NUM_THREADS", str(threads))
    op = oracle_from_solver(solver, shot)
    n = op.npts
    full = op.nsteps
    op.nsteps = min(full, 60)
    t0 = time.perf_counter()
    op.forward(fast=True)
    per_step = (time.perf_counter() - t0) / op.nsteps
    op.nsteps = int(max(60, min(full, seconds / (4.0 * per_step))))
    op.amp = op.amp[:op.nsteps]
    t0 = time.perf_counter()
    sim = op.forward(fast=True)["simdata"]
    op.migrate(0.1 * sim, fold=True, fast=True)
    t = time.perf_counter() - t0
    return {"value": 2.0 * n * op.nsteps / t / 1e9, "unit": "Gpt-updates/s", "cores": int(os.environ["OMP_NUM_THREADS"]),
            "kind": "port", "seconds": t,
            "sample": f"one shot's FP64 gradient on the {'x'.join(map(str, op.shape))} padded grid, "
                      f"{op.nsteps} of its {full} steps, order {op.order}, the oracle's forward + migrate loops "
                      f"(-O3 -fopenmp -ffast-math, node loops over {os.environ['OMP_NUM_THREADS']} threads; "
                      f"four propagations, the rate counts two)"}


TRAFFIC_FILES = {
    "c2": os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles", "traffic_k_step2d_layered2d.json"),
    "c4": os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles", "traffic_k_step3d_layered3d.json"),
}


def measured_traffic(shots, shape, tile_x, workload="c2"):
    """HBM bytes per launch of the forward and adjoint kernels from the
    committed rocprofv3 --pmc summary (FETCH_SIZE and WRITE_SIZE per
    dispatch, each scaled by the factor the same counter needs on a copy of
    known size), when it was measured on this workload and tile height;
    else nulls."""
    path = TRAFFIC_FILES[workload]
    try:
        with open(path) as f:
            t = json.load(f)
    except (OSError, ValueError):
        return {}
    if (t.get("shots") != shots or list(t.get("grid_padded", [])) != list(shape)
            or t.get("tile_x") != tile_x):
        return {}
    out = {"source": os.path.relpath(path, os.path.dirname(path) + "/..")}
    for k in ("forward", "adjoint"):
        d = t["kernels"][k]
        out[k] = d["fetch_kib"] * 1024 * t["fetch_factor"] + d["write_kib"] * 1024 * t["write_factor"]
    return out


def write_traffic(fetch_csv, write_csv, workload="c2"):
    """profiles/traffic_k_step2d_layered2d.json (c2) or
    traffic_k_step3d_layered3d.json (c4) from the counter files of the two
    `rocprofv3 --pmc FETCH_SIZE` / `--pmc WRITE_SIZE` runs of `bench.py
    --pmc-run`: per-dispatch averages of the forward (mode 1, with
    receivers: the largest grid) and adjoint (mode 4) kernels of the tile
    height most dispatched, and the factors that make each counter read the
    calibration copy's 262144 KiB (torch.add over 2^26 floats)."""
    import csv
    import collections
    import re

    def load(path, counter):
        disp = collections.OrderedDict()
        for r in csv.DictReader(open(path)):
            if r["Counter_Name"] != counter:
                continue
            d = disp.setdefault(int(r["Dispatch_Id"]), {"name": r["Kernel_Name"], "grid": int(r["Grid_Size"]),
                                                         "v": 0.0})
            d["v"] += float(r["Counter_Value"])
        return list(disp.values())

    if workload == "c4":
        shots, shape, kname = 8, (288, 288, 288), "k_step3d"
        pat = re.compile(r"pa::k_step3d<float, 4, (\d), true>")
    else:
        shots, shape, kname = 16, (1041, 341), "k_step2d"
        pat = re.compile(r"pa::k_step2d<float, (\d+), 4, (\d), false>")
    out = {}
    for key, path, counter in (("fetch", fetch_csv, "FETCH_SIZE"), ("write", write_csv, "WRITE_SIZE")):
        ds = load(path, counter)
        cal = [d["v"] for d in ds if "_add<float>" in d["name"] and d["grid"] == 2 ** 24]
        step = collections.defaultdict(list)
        for d in ds:
            m = pat.search(d["name"])
            if m and workload == "c4":
                step[(16, int(m.group(1)))].append(d)
            elif m:
                step[(int(m.group(1)), int(m.group(2)))].append(d)
        tx = max({k[0] for k in step}, key=lambda t: sum(len(v) for k, v in step.items() if k[0] == t))
        fwd = step[(tx, 1)]
        gmax = max(d["grid"] for d in fwd)
        fwd = [d["v"] for d in fwd if d["grid"] == gmax]
        adj = [d["v"] for d in step[(tx, 4)]]
        out[key] = {"cal": sum(cal) / len(cal), "tx": tx, "fwd": (sum(fwd) / len(fwd), len(fwd)),
                    "adj": (sum(adj) / len(adj), len(adj))}
    f, w = out["fetch"], out["write"]
    tx = f["tx"]
    wflag = " --workload c4" if workload == "c4" else ""
    doc = {
        "workload": (f"3D layered, {'x'.join(map(str, shape))} padded, {shots} shots, order 8, FP32 "
                     "(bench.py --workload c4 --pmc-run, 12 slots)" if workload == "c4" else
                     f"2D layered, {shape[0]}x{shape[1]} padded, {shots} shots, order 8, FP32 "
                     "(bench.py --pmc-run, 40 slots)"),
        "shots": shots, "grid_padded": list(shape), "tile_x": tx,
        "commands": ([] if workload == "c4" else [
            "PYSIT_AMD_TUNE_CACHE=prof/tune.json python3 bench.py  (the launch configuration chosen)"]) + [
            "PYSIT_AMD_TUNE_CACHE=prof/tune.json rocprofv3 --pmc FETCH_SIZE -d prof/pmcf -o run "
            f"--output-format csv -- python3 bench.py{wflag} --pmc-run --steps 1 --warmup 0",
            "PYSIT_AMD_TUNE_CACHE=prof/tune.json rocprofv3 --pmc WRITE_SIZE -d prof/pmcw -o run "
            f"--output-format csv -- python3 bench.py{wflag} --pmc-run --steps 1 --warmup 0",
            f"python3 bench.py{wflag} --write-traffic prof/pmcf/run_counter_collection.csv "
            "prof/pmcw/run_counter_collection.csv"],
        "calibration": {"kernel": "torch.add(x, 1.0, out=y) over 2^26 float32 (reads and writes 262144 KiB)",
                        "fetch_kib": f["cal"], "write_kib": w["cal"]},
        "fetch_factor": round(262144.0 / f["cal"], 4), "write_factor": round(262144.0 / w["cal"], 4),
        "kernels": {
            "forward": {"name": f"k_step3d<float,4,1>" if workload == "c4" else f"k_step2d<float,{tx},4,1>",
                        "dispatches": f["fwd"][1],
                        "fetch_kib": round(f["fwd"][0], 1), "write_kib": round(w["fwd"][0], 1)},
            "adjoint": {"name": f"k_step3d<float,4,4>" if workload == "c4" else f"k_step2d<float,{tx},4,4>",
                        "dispatches": f["adj"][1],
                        "fetch_kib": round(f["adj"][0], 1), "write_kib": round(w["adj"][0], 1)}},
    }
    with open(TRAFFIC_FILES[workload], "w") as fh:
        json.dump(doc, fh, indent=1)
        fh.write("\n")
    print(json.dumps(doc))


def run_c1(args):
    """The reference's own CPU case: the 2D horizontal reflector (91 x 71,
    dx 0.01, order 4, T = 1.5, PML 0.1, one Ricker source, 91 receivers) in
    FP64 through PySIT's API on the device: forward_model with
    simdata and dWaveOp, then migrate_shot of the residual against the true
    model's data, per step of the bench.  Beside it, the same gradient on the
    host through the oracle's loops (FP64, all host threads), and the device
    results against it.  Prints one JSON line."""
    import torch
    import pysit_amd as pa
    from pysit_amd.workloads import horizontal_reflector_2d
    from tests.problems import oracle_from_solver
    m, shots, solver, model = horizontal_reflector_2d()
    pa.generate_seismic_data(shots, solver, model)
    X, Z = m.mesh_coords()
    m0 = solver.ModelParameters(m, {"C": (1.0 + 0.3 * np.exp(-((Z - 0.45) / 0.02) ** 2)).reshape(-1, 1)})
    tm = pa.TemporalModeling(solver)
    shot = shots[0]

    def gradient():
        rv = tm.forward_model(shot, m0, 1, return_parameters=["simdata", "dWaveOp"])
        r = shot.receivers.interpolate_data(solver.ts()) - rv["simdata"]
        return rv["simdata"], r, tm.migrate_shot(shot, m0, r, 1, dWaveOp=rv["dWaveOp"])

    for _ in range(args.warmup):
        gradient()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        sim, r, g = gradient()
    torch.cuda.synchronize()
    t = (time.perf_counter() - t0) / args.steps
    shape = tuple(m.shape(include_bc=True, as_grid=True))
    n, nt = int(np.prod(shape)), solver.nsteps
    solver.model_parameters = m0
    op = oracle_from_solver(solver, shot)
    ref = op.forward()
    grad_ref = op.migrate(r)

    def rel(a, b):
        return float(np.linalg.norm(np.asarray(a).reshape(-1) - np.asarray(b).reshape(-1)) / np.linalg.norm(b))
    result = {
        "metric": "C1 forward_model + migrate_shot gradient Gpt-updates/s (FP64, PySIT API, one shot)",
        "value": 2.0 * n * nt / t / 1e9, "unit": "Gpt-updates/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": t * 1e3, "higher_is_better": True, "dtype": "f64",
        "data": "the reference's horizontal-reflector case (closed-form model), observed data generated in it; "
                "gradient at the reflector of 1.3",
        "config": {"workload": f"2D horizontal reflector, 91x71 ({shape[0]}x{shape[1]} padded), order 4, PML 0.1, "
                               f"T 1.5 (nt {nt} at the start model's dt), FP64",
                   "nt": nt, "grid_padded": list(shape)},
        "vs_oracle": {"traces_rel_l2": rel(sim, ref["simdata"]), "gradient_rel_l2": rel(g.data, grad_ref)},
        "residency": f"the state ({7 * n * 8 / 2**20:.1f} MiB of FP64 fields) and the dWaveOp history "
                     f"({nt * n * 8 / 2**20:.0f} MiB) sit on the chip or in the 256 MB Infinity Cache; "
                     f"{n} nodes are bound by a step's latency, not by HBM",
    }
    if not args.no_cpu:
        cpu = cpu_gradient(solver, shot, 20.0)
        result["cpu_baseline"] = cpu
        result["vs_cpu"] = result["value"] / cpu["value"]
    print(json.dumps(result), flush=True)


def run_uneven(args):
    """64 shots of seeded random aperture (300-1001 columns of the layered
    model) and length (1500-4000 steps) in one batch: the gradient of
    0.5 dt ||d||^2 (residual = the traces), checkpointed when the dWaveOp
    history exceeds the memory budget.  Prints one JSON line with the
    aggregate rate and the per-shot FP32 errors against the FP64 device path
    (itself matched to the FP64 oracle to 1e-10 by the GPU tests)."""
    import torch
    from pysit_amd.device import DeviceBatch
    from pysit_amd.workloads import uneven_2d
    t0 = time.perf_counter()
    geos, model, deltas, dt, meta = uneven_2d(n_shots=args.shots if args.shots != 16 else 64)
    t_setup = time.perf_counter() - t0
    work = sum(2.0 * g.npts * g.nt for g in geos)
    budget = int(args.memory_budget_gb * 2 ** 30) if args.memory_budget_gb else None

    def gradient(dtype, res=None, timed=False):
        b = DeviceBatch(geos, model, deltas, dt, 8, dtype=dtype, memory_budget=budget)
        if res is None:
            tr = b.forward(keep_dw=False)
            res = [t.clone() for t in tr]
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        reps = (args.warmup + args.steps) if timed else 1
        times = []
        for i in range(reps):
            torch.cuda.synchronize()
            ev[0].record()
            tr = b.forward(keep_dw=True)
            b.migrate(res)
            ev[1].record()
            torch.cuda.synchronize()
            if i >= reps - (args.steps if timed else 1):
                times.append(ev[0].elapsed_time(ev[1]) * 1e-3)
        imgs = [b.image(i).cpu().numpy().reshape(-1).copy() for i in range(b.n_shots)]
        trs = [t.cpu().numpy().copy() for t in tr]
        K = b.K
        del b, tr
        torch.cuda.empty_cache()
        return res, imgs, trs, sum(times) / len(times), K

    res, im32, tr32, t32, K = gradient(np.float32, timed=True)
    res64 = [r.to(torch.float64) for r in res]
    _, im64, tr64, t64, K64 = gradient(np.float64, res=res64)

    def rel(a, b):
        nb = np.linalg.norm(b)
        return float(np.linalg.norm(a - b) / nb) if nb > 0 else 0.0

    ge = [rel(a, b) for a, b in zip(im32, im64)]
    te = [rel(a, b) for a, b in zip(tr32, tr64)]
    value = work / t32 / 1e9
    print(json.dumps({
        "metric": "C3 aggregate fwd+adjoint gradient Gpt-updates/s (uneven shots, one batch)",
        "value": value, "unit": "Gpt-updates/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": t32 * 1e3, "higher_is_better": True, "dtype": "f32", "data": "synthetic",
        "config": {"workload": f"{len(geos)} shots, aperture 300-1001 columns of the 1001x301 layered model, "
                               f"nt 1500-4000, order 8, PML 20, FP32",
                   "shots": len(geos), "work_gpt": work / 1e9, "dwaveop_segment": K,
                   "max_nt": max(g.nt for g in geos), "total_nodes": sum(g.npts for g in geos)},
        "fp64": {"seconds": t64, "dwaveop_segment": K64},
        "accuracy_vs_fp64": {"gradient_rel_l2_max": max(ge), "gradient_rel_l2_median": float(np.median(ge)),
                             "traces_rel_l2_max": max(te), "traces_rel_l2_median": float(np.median(te))},
        "host_setup_s": t_setup}), flush=True)


def run_3d(args):
    """The 3D case: 256^3 nodes at dx = 12.5 m (288^3 padded with 16 PML
    cells per side), velocities 1500-4000 m/s in seeded layers with a -10 %
    Gaussian anomaly (radius 400 m), 8 Ricker sources (6 Hz) in a line at 25 m
    depth, a 64 x 64 receiver patch at 25 m, nt = 2000 at the CFL step, FP32,
    order 8, in km and km/s (the 3D PML of the reference's step is stable in
    these units and not in m and m/s, see workloads.layered_3d).  One step is the gradient of 0.5 dt ||d||^2 (residual = the
    traces) over all 8 shots in one batch; the dWaveOp history does not fit,
    so the forward keeps checkpoints and the adjoint recomputes each segment
    (segment length from 80 % of free HBM).  value = 2 sum N nt / s, the
    recompute not counted.  FP32 against FP64 is measured on the first shot
    alone (eight FP64 shots do not fit a one-level checkpoint schedule in
    288 GB).  Prints one JSON line."""
    import torch
    from pysit_amd.device import DeviceBatch
    from pysit_amd.modeling import TemporalModeling
    from pysit_amd.workloads import layered_3d
    if args.pmc_run:
        # calibration: y = x + 1 over 2^26 floats reads and writes exactly 256 MiB
        x = torch.ones(2 ** 26, dtype=torch.float32, device="cuda")
        y = torch.empty_like(x)
        for _ in range(3):
            torch.add(x, 1.0, out=y)
        torch.cuda.synchronize()
        del x, y
        if args.nt == 3000:
            args.nt = 12
    t0 = time.perf_counter()
    nt = args.nt if args.nt != 3000 else 2000
    mesh, shots, solver, model = layered_3d(n=256, n_shots=8, nt=nt)
    tm = TemporalModeling(solver, autotune=False)
    geos = [tm.geometry(sh) for sh in shots]
    t_setup = time.perf_counter() - t0
    shape = tuple(mesh.shape(include_bc=True, as_grid=True))
    npts = int(np.prod(shape))
    npml = pml_nodes(shape, mesh.pad_widths())
    model_u = solver.unpadded_model()
    budget = int(args.memory_budget_gb * 2 ** 30) if args.memory_budget_gb else None

    def gradient(b, res, timed):
        reps = (args.warmup + args.steps) if timed else 1
        times = []
        for i in range(reps):
            keep = timed and i == reps - 1
            b.timer = {} if keep else None
            torch.cuda.synchronize()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            b.forward(keep_dw=True)
            b.migrate(res)
            e1.record()
            torch.cuda.synchronize()
            if i >= reps - (args.steps if timed else 1):
                times.append(e0.elapsed_time(e1) * 1e-3)
            print(f"[c4] gradient {i + 1}/{reps}: {times[-1] if times else e0.elapsed_time(e1) * 1e-3:.2f} s, "
                  f"segment {b.K}", file=sys.stderr, flush=True)
        return sum(times) / len(times)

    def avg_us(timer, mode):
        tot = sum(a.elapsed_time(e) for a, e, _ in timer.get(mode, []))
        n = sum(c for _, _, c in timer.get(mode, []))
        return tot * 1e3 / max(n, 1), n

    b = DeviceBatch(geos, model_u, mesh.deltas, solver.dt, 8, dtype=np.float32, memory_budget=budget)
    b32_window = bool(b.ic_window)
    res = [t.clone() for t in b.forward(keep_dw=False)]
    if args.pmc_run:
        b.forward(keep_dw=True)
        b.migrate(res)
        torch.cuda.synchronize()
        print(json.dumps({"pmc_run": "done", "nt": nt, "shots": len(shots), "tile_x": b.tile_x}), flush=True)
        return
    t32 = gradient(b, res, True)
    timer = b.timer
    adj_us, n_adj = avg_us(timer, 2)
    fwd_us, n_fwd = avg_us(timer, 1)
    b_fwd, b_adj = algorithmic_bytes([(npts, npml)] * len(shots), 4, dim=3)
    traffic = measured_traffic(len(shots), shape, b.tile_x, workload="c4")
    K = b.K
    img32 = b.image(0).cpu().numpy().reshape(-1).copy()
    tr32 = res[0].cpu().numpy().copy()
    del b
    torch.cuda.empty_cache()
    acc = None
    if not args.no_accuracy:
        b32 = DeviceBatch(geos[:1], model_u, mesh.deltas, solver.dt, 8, dtype=np.float32, memory_budget=budget)
        r32 = [t.clone() for t in b32.forward(keep_dw=False)]
        gradient(b32, r32, False)
        i32 = b32.image(0).cpu().numpy().reshape(-1).copy()
        del b32
        torch.cuda.empty_cache()
        b64 = DeviceBatch(geos[:1], model_u, mesh.deltas, solver.dt, 8, dtype=np.float64, memory_budget=budget)
        r64 = [r32[0].to(torch.float64)]
        tr64 = b64.forward(keep_dw=False)[0].cpu().numpy().copy()
        gradient(b64, r64, False)
        i64 = b64.image(0).cpu().numpy().reshape(-1).copy()
        del b64
        torch.cuda.empty_cache()

        def rel(a, c):
            return float(np.linalg.norm(a - c) / np.linalg.norm(c))
        acc = {"traces_rel_l2": rel(r32[0].cpu().numpy(), tr64), "gradient_rel_l2": rel(i32, i64),
               "note": "first shot, FP32 against the FP64 device path on the same residual"}
    work = 2.0 * npts * nt * len(shots)
    value = work / t32 / 1e9
    ach = b_adj / (adj_us * 1e-6) / 1e9
    print(json.dumps({
        "metric": "C4 3D fwd+adjoint gradient Gpt-updates/s (8 shots, checkpointed)",
        "value": value, "unit": "Gpt-updates/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": t32 * 1e3, "higher_is_better": True, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "3D layered + anomaly, 256^3 (288^3 padded), dx=12.5 m, order 8, PML 16, 8 shots, "
                               "64x64 receivers, FP32, checkpointed; units km, km/s, s",
                   "shots": len(shots), "nt": nt, "grid_padded": list(shape), "dwaveop_segment": K,
                   "checkpoints": -(-nt // K)},
        "roofline": {"bound": "hbm", "achieved": ach, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": ach / HBM_PEAK_GBS, "traffic": traffic.get("adjoint"),
                     "kernel": ("k_step3d<float,4,4> (adjoint + imaging, FP32 window sums into FP64)"
                                if b32_window else "k_step3d<float,4,2> (adjoint + FP64 imaging)"),
                     "bytes_per_launch": b_adj, "avg_launch_us": adj_us, "launches": n_adj},
        "forward_kernel": {"kernel": "k_step3d<float,4,1> (recompute + dWaveOp store)", "avg_launch_us": fwd_us,
                           "achieved_gbs": b_fwd / (fwd_us * 1e-6) / 1e9, "bytes_per_launch": b_fwd,
                           "launches": n_fwd, "traffic": traffic.get("forward")},
        "traffic_source": traffic.get("source"),
        "gradient_roofline_frac": value * 1e9 * (b_fwd + b_adj) / (2 * npts * len(shots)) / 1e9 / HBM_PEAK_GBS,
        "accuracy_vs_fp64": acc, "host_setup_s": t_setup}), flush=True)


def run_fwi(args):
    """The 2D FWI loop: 601 x 201 nodes at dx = 15 m (641 x 241 padded), the
    layered true model, its 300 m Gaussian smoothing as the start model, 32
    shots with 601 receivers, nt = 2500 at the true model's CFL step, order
    8; for each band (Ricker peaks 3, 5, 8 Hz) observed data from the true
    model and --fwi-iterations LBFGS iterations (memory 10) of
    TemporalLeastSquares with the backtracking line search.  Run in FP32
    (timed: value = algorithmic grid-point updates of every forward, gradient
    and line-search evaluation over the wall time of the loop, host work
    included) and again in FP64 on the device, whose gradients match the FP64
    oracle to 1e-10 in the GPU tests; prints one JSON line."""
    import torch
    from pysit_amd.workloads import fwi_2d, multiband_fwi, model_error
    bands = tuple(float(f) for f in args.fwi_bands.split(","))
    out = {}
    for prec in ("single", "double"):
        if prec == "double" and args.no_accuracy:
            break
        mesh, solver, true_model, start_model = fwi_2d(precision=prec)
        print(f"[c5] {prec}: bands {bands}, {args.fwi_iterations} iterations each", file=sys.stderr, flush=True)
        t0 = time.perf_counter()
        model, reports = multiband_fwi(mesh, solver, true_model, start_model, bands=bands,
                                       iterations=args.fwi_iterations, verbose=True, sync=torch.cuda.synchronize,
                                       log=sys.stderr)
        torch.cuda.synchronize()
        out[prec] = {"model": model, "reports": reports, "seconds": time.perf_counter() - t0,
                     "start_error": model_error(start_model, true_model), "true": true_model}
        torch.cuda.empty_cache()
    s32 = out["single"]
    updates = sum(r["updates"] for r in s32["reports"])
    value = updates / s32["seconds"] / 1e9

    def band_summary(reports):
        return [{"f0_hz": r["f0_hz"], "objective_first": r["objective"][0], "objective_final": r["objective"][-1],
                 "misfit_reduction": r["misfit_reduction"], "model_error_start": r["model_error_start"],
                 "model_error_final": r["model_error_final"],
                 "model_error_upper_third_start": r["model_error_shallow_start"],
                 "model_error_upper_third_final": r["model_error_shallow_final"], "evaluations": r["evaluations"],
                 "gradients": r["gradients"], "seconds": r["seconds"]} for r in reports]
    line = {
        "metric": "C5 multi-band FWI loop Gpt-updates/s (forward, gradient and line-search evaluations, "
                  "host work included)",
        "value": value, "unit": "Gpt-updates/s", "n_gpus": 1, "steps": len(bands) * args.fwi_iterations,
        "warmup": 0, "ms_per_step": s32["seconds"] * 1e3 / (len(bands) * args.fwi_iterations),
        "higher_is_better": True, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "2D FWI, 601x201 (641x241 padded), dx=15 m, order 8, PML 20, 32 shots, "
                               "601 receivers, nt 2500 at the true model's CFL dt, layered + random field true "
                               "model, 300 m smoothed start, LBFGS memory 10, backtracking line search",
                   "bands_hz": list(bands), "iterations_per_band": args.fwi_iterations},
        "fp32": {"seconds": s32["seconds"], "updates_gpt": updates / 1e9,
                 "model_error_start": s32["start_error"],
                 "model_error_final": model_error(s32["model"], s32["true"]),
                 "model_error_upper_third_start": s32["reports"][0]["model_error_shallow_start"],
                 "model_error_upper_third_final": s32["reports"][-1]["model_error_shallow_final"],
                 "bands": band_summary(s32["reports"])},
    }
    if "double" in out:
        s64 = out["double"]
        c32, c64 = np.asarray(s32["model"].C).ravel(), np.asarray(s64["model"].C).ravel()
        o32 = np.concatenate([r["objective"] for r in s32["reports"]])
        o64 = np.concatenate([r["objective"] for r in s64["reports"]])
        n = min(len(o32), len(o64))
        line["fp64"] = {"seconds": s64["seconds"], "model_error_final": model_error(s64["model"], s64["true"]),
                        "bands": band_summary(s64["reports"])}
        line["fp32_vs_fp64"] = {
            "final_model_rel_l2": float(np.linalg.norm(c32 - c64) / np.linalg.norm(c64)),
            "objective_history_max_rel": float(np.max(np.abs(o32[:n] - o64[:n]) / np.abs(o64[:n])))}
    print(json.dumps(line), flush=True)


def main():
    args = parse()
    if args.write_traffic:
        write_traffic(*args.write_traffic, workload=args.workload)
        return
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported here (more GPUs would each run "
              f"a share of the shots in a process of their own and sum the images and misfits)", file=sys.stderr)
        sys.exit(2)
    import torch
    import pysit_amd as pa
    from pysit_amd.torch_fn import ShotProblem, ShotTraces
    from pysit_amd.workloads import layered_2d
    if args.workload == "c1":
        run_c1(args)
        return
    if args.workload == "c3":
        run_uneven(args)
        return
    if args.workload == "c4":
        run_3d(args)
        return
    if args.workload == "c5":
        run_fwi(args)
        return
    if args.pmc_run:
        # calibration: y = x + 1 over 2^26 floats reads and writes exactly 256 MiB
        x = torch.ones(2 ** 26, dtype=torch.float32, device="cuda")
        y = torch.empty_like(x)
        for _ in range(3):
            torch.add(x, 1.0, out=y)
        torch.cuda.synchronize()
        del x, y
        if args.nt == 3000:
            args.nt = 40

    dev = torch.device("cuda", 0)
    mesh, shots, solver, model = layered_2d(n_shots=args.shots, nt=args.nt)
    shots = shots[:args.shots]
    nx, nz = mesh.shape(as_grid=True)
    shape = tuple(mesh.shape(include_bc=True, as_grid=True))
    pads = mesh.pad_widths()
    npts = int(np.prod(shape))
    nt = solver.nsteps
    dt = solver.dt
    budget = int(args.memory_budget_gb * 2 ** 30) if args.memory_budget_gb else None

    # observed data from the layered model; the gradient is taken at an FWI
    # start model: the layered model Gaussian-smoothed (sigma 300 m) and
    # rescaled to the same maximum velocity (so dt and nt are unchanged)
    from scipy.ndimage import gaussian_filter
    v_true = model.C.reshape(nx, nz)
    v0 = gaussian_filter(v_true, sigma=300.0 / mesh.deltas[0], mode="nearest")
    v0 *= v_true.max() / v0.max()
    tm = pa.TemporalModeling(solver, memory_budget=budget, tile_x=args.tile_x)
    d_obs = torch.from_numpy(np.stack(tm.forward_model_batch(shots, model))).to(dev)
    tm.last_batch = None

    m = torch.from_numpy(v0 ** -2.0).to(dev).requires_grad_(True)
    # launch configuration: autotuned (a counter run should read the choice of
    # a plain run from PYSIT_AMD_TUNE_CACHE: counters distort the tuner's timings)
    problem = ShotProblem(solver, shots, memory_budget=budget, tile_x=args.tile_x)

    last = {}

    def gradient(prob, mm=None):
        mm = m if mm is None else mm
        if mm.grad is not None:
            mm.grad = None
        tr = ShotTraces.apply(mm, prob)
        loss = 0.5 * dt * ((tr - d_obs[:tr.shape[0]]) ** 2).sum()
        loss.backward()
        last["traces"] = tr.detach()
        return loss

    for _ in range(args.warmup):
        gradient(problem)
    torch.cuda.synchronize()
    problem.timer = {}
    t0 = time.perf_counter()
    for _ in range(args.steps):
        loss = gradient(problem)
    torch.cuda.synchronize()
    t_step = (time.perf_counter() - t0) / args.steps
    timer, problem.timer = problem.timer, None
    problem.batch.timer = None

    updates = 2.0 * npts * nt * len(shots)
    value = updates / t_step / 1e9
    segment = problem.batch.K
    gnorm = float(m.grad.norm())

    # per-kernel average launch duration over the timed region (HIP events)
    def avg_ms(mode):
        tot = sum(s.elapsed_time(e) for s, e, _ in timer.get(mode, []))
        n = sum(c for _, _, c in timer.get(mode, []))
        return tot / max(n, 1), n

    fwd_ms, n_fwd = avg_ms(1)
    adj_ms, n_adj = avg_ms(2)
    traffic = measured_traffic(len(shots), shape, problem.batch.tile_x)
    itemsize = 4 if solver.dtype == np.single else 8
    npml = pml_nodes(shape, pads)
    b_fwd, b_adj = algorithmic_bytes([(npts, npml)] * len(shots), itemsize)
    resident = problem.batch.resident_tables()
    if resident is not None:
        # the fields stay on the chip: a step moves the dWaveOp history alone
        b_fwd = b_adj = npts * len(shots) * itemsize
        traffic = {}
    ach_adj = b_adj / (adj_ms * 1e-3) / 1e9
    ach_fwd = b_fwd / (fwd_ms * 1e-3) / 1e9
    grad_bytes = nt * (b_fwd + b_adj)

    result = {
        "metric": METRIC,
        "value": value,
        "unit": "Gpt-updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": t_step * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic (seeded layered model, Ricker sources; gradient at its 300 m Gaussian-smoothed start model)",
        "config": {"workload": "2D layered, 1001x301 (1041x341 padded), dx=10 m, order 8, PML 20, "
                               f"{len(shots)} shots x 1001 receivers, nt={nt}, FP32, batched fused launches, "
                               f"dWaveOp segment {segment} of {nt} slots",
                   "grid_padded": list(shape), "shots": len(shots), "nt": nt, "order": 8,
                   "tile_x": problem.batch.tile_x, "tile_order": problem.batch.tile_order,
                   "graph_steps": problem.batch.graph_steps},
        "roofline": {"bound": "hbm", "achieved": ach_adj, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": ach_adj / HBM_PEAK_GBS, "traffic": traffic.get("adjoint"),
                     "kernel": (f"k_step2d<float,{problem.batch.tile_x},4,4> (adjoint + imaging, FP32 window "
                                "sums into FP64)" if problem.batch.ic_window else
                                f"k_step2d<float,{problem.batch.tile_x},4,2> (adjoint + FP64 imaging)"),
                     "bytes_per_launch": b_adj, "avg_launch_us": adj_ms * 1e3, "launches": n_adj},
        "forward_kernel": {"kernel": f"k_step2d<float,{problem.batch.tile_x},4,1> (forward + dWaveOp store)",
                           "achieved_gbs": ach_fwd, "frac": ach_fwd / HBM_PEAK_GBS,
                           "avg_launch_us": fwd_ms * 1e3, "bytes_per_launch": b_fwd, "launches": n_fwd,
                           "traffic": traffic.get("forward")},
        "traffic_source": traffic.get("source"),
        "gradient_roofline_frac": grad_bytes / t_step / 1e9 / HBM_PEAK_GBS,
        "bytes_per_update": grad_bytes / updates,
        "residency": (f"HBM: the {len(shots)} shots' state ({problem.batch.state_bytes() / 2**20:.0f} MiB) and "
                      f"the dWaveOp store ({segment * problem.batch.total_n * 4 / 2**30:.1f} GiB) exceed the "
                      f"256 MB Infinity Cache"),
        "misfit": float(loss.detach()), "grad_norm": gnorm,
    }

    if resident is not None:
        # neither memory nor one unit (counters, profiles/k_resident2d_layered2d_16shots.md)
        result["roofline"].update(bound="latency of a step on the chip (vector instructions and waits of the PML rows)",
                                  kernel="k_resident2d<float,4,4> (adjoint + imaging, fields on the chip; per step)")
        result["forward_kernel"]["kernel"] = "k_resident2d<float,4,1> (forward + dWaveOp store, fields on the chip; " \
                                             "per step)"
        result["residency"] = (f"LDS and registers: the shots' fields, {len(resident.group_lds)} groups of shots, "
                               f"{resident.n_strips} strips; HBM: the dWaveOp store "
                               f"({segment * problem.batch.total_n * 4 / 2**30:.1f} GiB)")

    if args.ckpt_budget_gb and not (args.profile_run or args.pmc_run):
        # the same gradient with the dWaveOp history checkpointed: the budget
        # holds a store of K slots and the checkpoints, and the adjoint
        # recomputes each segment's dWaveOp (those launches are not counted
        # in the rate).  The FP32 imaging windows follow the slots, so the
        # gradient equals the store-all one bit for bit
        g_all = m.grad.detach().clone()
        problem.batch = None
        torch.cuda.empty_cache()
        ck_budget = int(args.ckpt_budget_gb * 2 ** 30)
        ck = ShotProblem(solver, shots, memory_budget=ck_budget, tile_x=args.tile_x)
        for _ in range(args.warmup):
            gradient(ck)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            gradient(ck)
        torch.cuda.synchronize()
        t_ck = (time.perf_counter() - t0) / args.steps
        b = ck.batch
        result["checkpointed"] = {
            "value": updates / t_ck / 1e9, "unit": "Gpt-updates/s", "ms_per_step": t_ck * 1e3,
            "memory_budget_gib": args.ckpt_budget_gb, "dwaveop_segment": b.K, "levels": [int(v) for v in b.levels],
            "schedule": "binomial" if b.snaps is not None else "nested segments",
            "gradient_vs_store_all_rel_l2": float(torch.linalg.norm((m.grad - g_all).double())
                                                  / torch.linalg.norm(g_all.double())),
            "gradient_roofline_frac": grad_bytes / t_ck / 1e9 / HBM_PEAK_GBS,
            "note": "rate counts 2 N nt per shot; the dWaveOp recompute launches are extra work"}
        ck.batch = None
        del ck, b
        torch.cuda.empty_cache()
    if args.pmc_run:
        b = problem.batch
        print(json.dumps({"pmc_run": "done", "nt": nt, "shots": len(shots), "tile_x": b.tile_x,
                          "tile_order": b.tile_order, "graph_steps": b.graph_steps}), flush=True)
        return
    if not (args.no_accuracy or args.profile_run):
        # the same gradient through the FP64 device path (matched to the FP64
        # oracle to 1e-10 by the GPU tests) as the reference for the FP32 errors
        g32 = m.grad.detach().clone()
        tr32 = last["traces"].clone()
        problem.batch = None
        torch.cuda.empty_cache()
        mesh64, shots64, solver64, model64 = layered_2d(n_shots=args.shots, nt=args.nt, precision="double")
        m64 = m.detach().to(torch.float64).clone().requires_grad_(True)
        prob64 = ShotProblem(solver64, shots64[:args.shots], memory_budget=budget)
        loss64 = gradient(prob64, m64)
        g64 = m64.grad.detach()

        def rel(a, b):
            return float(torch.linalg.norm(a - b) / torch.linalg.norm(b))

        result["accuracy_vs_fp64"] = {
            "traces_rel_l2": rel(tr32, last["traces"]), "gradient_rel_l2": rel(g32.to(torch.float64), g64),
            "misfit_rel": abs(float(loss.detach()) - float(loss64.detach())) / float(loss64.detach()),
            "note": "FP32 path vs the FP64 device path on the same inputs; the reference's own FP32 step "
                    "arithmetic is 1.9e-4 off its FP64 traces on one of these shots (3000 steps)"}
        # the loss keeps its graph, whose node keeps the batch and its store
        del prob64, loss64, m64, g64
        torch.cuda.empty_cache()
    if not (args.no_plain or args.profile_run):
        plain = [ShotProblem(solver, [s], memory_budget=budget, tile_x=args.tile_x) for s in shots]
        for p in plain[:1]:
            gradient(p)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for p in plain:
            gradient(p)
            p.batch = None
        torch.cuda.synchronize()
        t_plain = time.perf_counter() - t0
        result["plain"] = {"value": updates / t_plain / 1e9, "ms_per_gradient": t_plain * 1e3,
                           "form": "one shot per launch, same kernels, 16 sequential shot gradients"}
        result["batched_vs_plain"] = t_plain / t_step
        if "checkpointed" in result:
            result["checkpointed"]["vs_plain"] = t_plain / (result["checkpointed"]["ms_per_step"] * 1e-3)

    if not (args.no_cpu or args.profile_run):
        kp = solver.kernel_pml()
        result["cpu_baseline"] = cpu_baseline(shape, kp, dt, mesh.deltas, args.cpu_seconds)
        result["cpu_baseline"]["gradient"] = cpu_gradient(solver, shots[len(shots) // 2], args.cpu_seconds * 4)
    if not (args.no_3d or args.profile_run):
        # the 3D checkpointed gradient (--workload c4, one timed gradient) in
        # a child process with the device memory to itself
        import gc
        # the last loss keeps its autograd graph, whose node keeps the
        # batch and its dWaveOp store: release them before the child runs
        problem.batch = None
        loss = None
        last.clear()
        gc.collect()
        torch.cuda.empty_cache()
        free, total = torch.cuda.mem_get_info()
        result["c4_3d"] = run_child_3d()
        result["c4_3d"]["device_free_gib_at_start"] = free / 2 ** 30
    print(json.dumps(result), flush=True)


def run_child_3d():
    """--workload c4 --steps 1 --warmup 0 --no-cpu in a child process; its
    JSON line, condensed (or the failure)."""
    import subprocess
    cmd = [sys.executable, os.path.abspath(__file__), "--workload", "c4", "--steps", "1", "--warmup", "0",
           "--no-cpu"]
    print("[c2] 3D checkpointed gradient in a child process", file=sys.stderr, flush=True)
    try:
        p = subprocess.run(cmd, capture_output=True, text=True, timeout=900)
    except subprocess.TimeoutExpired:
        return {"error": "timed out after 900 s"}
    lines = [l for l in p.stdout.splitlines() if l.startswith("{")]
    if p.returncode != 0 or not lines:
        return {"error": f"exit {p.returncode}", "stderr_tail": p.stderr[-800:]}
    d = json.loads(lines[-1])
    keep = ("metric", "value", "unit", "ms_per_step", "steps", "warmup", "gradient_roofline_frac",
            "accuracy_vs_fp64", "config")
    out = {k: d[k] for k in keep if k in d}
    r = d.get("roofline", {})
    out["roofline"] = {k: r.get(k) for k in ("kernel", "achieved", "peak", "unit", "frac", "traffic",
                                              "avg_launch_us")}
    out["command"] = " ".join(["python3", "bench.py"] + cmd[2:])
    return out


if __name__ == "__main__":
    main()
