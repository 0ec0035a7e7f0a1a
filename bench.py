#!/usr/bin/env python3
"""Benchmark of the coupled surface/subsurface solver on one MI355X.

Workload (default): the 400x400x30 coupled run -- 1% slope + GRF topography, log-normal Ks,
20 mm/h rain for 3600 s then 3600 s recession, dt = 30 s, 240 steps -- solved three times from
the same synthetic inputs:
  * FP64 with the column-preconditioned PCG,
  * mixed precision (FP32 column-preconditioned PCG + FP64 residual refinement), and
  * the plain FP64 path (FP64 Jacobi-PCG, one launch per iteration), and
  * the mixed-precision form of that Jacobi-PCG (FP32 with FP64 reliable updates).
A step is one coupled time step (subsurface Picard solve + overland solve) over the whole
grid.  `value` is the mixed-precision throughput in 3D cell-steps/s; the FP64 and plain
throughputs, the speed-ups, and the head error of the mixed run against the FP64 run are in
the same line.

The dominant kernel's roofline comes from HIP events recorded by the library on its own
stream around every Krylov launch of the timed region.  The CPU baseline is the oracle
(FP64 C++/OpenMP restatement of the reference algorithm) timed on a bounded window of the
same workload, started from the GPU FP64 state at that step.

Usage: python bench.py [--steps K] [--warmup W] [--gpus 1]
       python bench.py --workload ensemble [--members M]   (the batched 256-member ensemble)
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "cell-steps/s and %HBM roofline, mixed vs FP64 at ≤1e-6 m head error"
HBM_PEAK = 8.0e12          # MI355X HBM3E, bytes/s


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=240)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--nx", type=int, default=400)
    ap.add_argument("--ny", type=int, default=400)
    ap.add_argument("--nz", type=int, default=30)
    ap.add_argument("--cpu-start", type=int, default=60)
    ap.add_argument("--cpu-steps", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-1thread-steps", type=int, default=1,
                    help="steps of the CPU window run again on one thread (0: skip)")
    ap.add_argument("--no-c1", action="store_true", help="skip the C1 run (32x32x20, 100 steps) on GPU and CPU")
    ap.add_argument("--only", choices=["both", "fp64", "mixed"], default="both")
    ap.add_argument("--refine-max", type=int, default=None, help="mixed: FP64 refinement sweeps per Picard iteration")
    ap.add_argument("--inner-tol", type=float, default=None, help="mixed: FP32 inner relative tolerance")
    ap.add_argument("--mixed-lin-tol", type=float, default=None, help="mixed: FP64 residual target")
    ap.add_argument("--tile-f64", default=None, metavar="TX,TY,KC",
                    help="SpMV tile of the FP64 solves instead of the autotuner's (profiler runs, whose "
                         "instrumentation distorts the tuning)")
    ap.add_argument("--tile-f32", default=None, metavar="TX,TY,KC", help="the same for the FP32 solves")
    ap.add_argument("--no-plain", action="store_true",
                    help="skip the plain FP64 Jacobi-PCG reference run (with --precond column)")
    ap.add_argument("--precond", choices=["jacobi", "column"], default="column",
                    help="subsurface PCG preconditioner (column: exact solve of each column's vertical "
                         "tridiagonal part, two-kernel recurrences with a column-solve kernel)")
    ap.add_argument("--krylov", choices=["one", "two"], default="one",
                    help="subsurface PCG: one launch per iteration (single-reduction recurrences) or the "
                         "two-kernel Hestenes-Stiefel form")
    ap.add_argument("--workload", choices=["coupled", "ensemble"], default="coupled",
                    help="ensemble: the batched 256-member ensemble (200 steps, mixed precision)")
    ap.add_argument("--members", type=int, default=256, help="ensemble: number of members")
    ap.add_argument("--no-graph", action="store_true",
                    help="ensemble: launch the Krylov batches eagerly instead of replaying a captured hipGraph")
    ap.add_argument("--prof-steps", type=int, default=3,
                    help="steps after the timed region run with kernel timestamps (roofline)")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="first run three plain 1 GiB device-to-device copies (for scaling HBM counters)")
    ap.add_argument("--trace-summary", metavar="KERNEL_TRACE_CSV", default=None,
                    help="summarise a rocprofv3 kernel trace (per kernel, launches that did work) and exit")
    ap.add_argument("--sq-summary", metavar="SQ_COUNTER_CSV", default=None,
                    help="occupancy and stall fractions per kernel from a rocprofv3 --pmc run of the eight "
                         "SQ counters in SQ_COUNTERS (counter_collection.csv); prints a table and exits")
    ap.add_argument("--pmc-summary", nargs=2, metavar=("FETCH_CSV", "WRITE_CSV"), default=None,
                    help="HBM bytes per working launch of each kernel from two rocprofv3 --pmc runs (FETCH_SIZE, "
                         "WRITE_SIZE counter_collection.csv), scaled by the same counters' reading of the 1 GiB "
                         "device-to-device copies of --calibrate-copy; prints JSON and exits")
    return ap.parse_args()


def trace_summary(path):
    """Per-kernel launch counts and average durations from a rocprofv3 kernel_trace.csv.
    Krylov kernels queued past the end of a solve return at once (a few us), and the SpMV launch
    that finds a solve converged only sums the partials (~10 us); those launches are split off:
    a launch did the full work when it took more than half the kernel's 90th-percentile
    duration."""
    import csv
    from collections import defaultdict
    dur = defaultdict(list)
    with open(path) as fh:
        for row in csv.DictReader(fh):
            dur[row["Kernel_Name"]].append(int(row["End_Timestamp"]) - int(row["Start_Timestamp"]))
    lines = ["| kernel | launches | did work | avg us (working) | avg us (all) | total ms |",
             "|---|---|---|---|---|---|"]
    for name, v in sorted(dur.items(), key=lambda kv: -sum(kv[1])):
        v = np.array(v, dtype=np.float64)
        work = v[v > 0.5 * np.percentile(v, 90)]
        short = name.replace("(anonymous namespace)::", "").split("(")[0]
        lines.append(f"| {short} | {len(v)} | {len(work)} | {work.mean() / 1e3:.2f} | {v.mean() / 1e3:.2f} | "
                     f"{v.sum() / 1e6:.1f} |")
    print("\n".join(lines[:22]))


def _kernel_short(name):
    return name.replace("(anonymous namespace)::", "").replace("dh::", "").split("(")[0].strip()


def pmc_summary(fetch_csv, write_csv):
    """Per-kernel HBM traffic per working launch: FETCH_SIZE and WRITE_SIZE (KiB per dispatch)
    times the factor that maps the counter's reading of a 1 GiB device-to-device copy (1 GiB read,
    1 GiB written) to 1 GiB; launches that did work are those above half the kernel's
    90th-percentile total (as in --trace-summary)."""
    import csv
    from collections import defaultdict

    def load(path, counter):
        vals = defaultdict(list)
        with open(path) as fh:
            for row in csv.DictReader(fh):
                if row["Counter_Name"] == counter:
                    vals[_kernel_short(row["Kernel_Name"])].append(float(row["Counter_Value"]))
        return vals
    fetch, write = load(fetch_csv, "FETCH_SIZE"), load(write_csv, "WRITE_SIZE")
    gib_kib = float(1 << 20)
    copies_f = sorted(fetch.get("__amd_rocclr_copyBuffer", []))[-3:]
    copies_w = sorted(write.get("__amd_rocclr_copyBuffer", []))[-3:]
    if len(copies_f) < 3 or len(copies_w) < 3 or min(copies_f) < 0.25 * gib_kib:
        raise SystemExit("no 1 GiB calibration copies in the counter files (profile with --calibrate-copy)")
    ff, fw = gib_kib / float(np.mean(copies_f)), gib_kib / float(np.mean(copies_w))
    out = {"calibration": {"fetch_factor": ff, "write_factor": fw,
                           "reference": f"three 1 GiB device-to-device copies: FETCH_SIZE {np.mean(copies_f):.0f} KiB, "
                                        f"WRITE_SIZE {np.mean(copies_w):.0f} KiB per copy"},
           "unit": "HBM bytes per working launch (FETCH_SIZE x fetch_factor + WRITE_SIZE x write_factor, KiB x 1024)"}
    for name in sorted(set(fetch) & set(write)):
        if name.startswith("__amd"):
            continue
        f, w = np.array(fetch[name]), np.array(write[name])
        if len(f) != len(w):
            continue
        tot = f * ff + w * fw
        work = tot > 0.5 * np.percentile(tot, 90)
        out[name] = {"launches": int(len(f)), "working": int(work.sum()),
                     "fetch_bytes": float(np.median(f[work]) * ff * 1024),
                     "write_bytes": float(np.median(w[work]) * fw * 1024),
                     "bytes_per_launch": float(np.median(tot[work]) * 1024)}
    print(json.dumps(out, indent=1))


SQ_COUNTERS = ["SQ_WAVES", "SQ_WAVE_CYCLES", "SQ_BUSY_CU_CYCLES", "SQ_WAIT_ANY", "SQ_ACTIVE_INST_ANY",
               "SQ_ACTIVE_INST_VMEM", "SQ_ACTIVE_INST_VALU", "SQ_ACTIVE_INST_LDS"]


def sq_summary(path):
    """Occupancy and stall fractions per kernel from one rocprofv3 --pmc run of SQ_COUNTERS:
    per dispatch, waves per SIMD = SQ_WAVE_CYCLES / SQ_BUSY_CU_CYCLES and the fractions of the
    waves' resident time spent waiting or issuing (over SQ_WAVE_CYCLES); the median over the
    dispatches that did work (SQ_WAVE_CYCLES above half the kernel's 90th percentile)."""
    import csv
    from collections import defaultdict
    disp, name = defaultdict(dict), {}
    with open(path) as fh:
        for r in csv.DictReader(fh):
            d = r.get("Dispatch_Id") or r.get("Correlation_Id")
            disp[d][r["Counter_Name"]] = disp[d].get(r["Counter_Name"], 0.0) + float(r["Counter_Value"])
            name[d] = _kernel_short(r["Kernel_Name"])
    by = defaultdict(list)
    for d, c in disp.items():
        if all(k in c for k in SQ_COUNTERS):
            by[name[d]].append(c)
    print("| kernel | dispatches (working) | waves per SIMD | wave time waiting | issuing any | VMEM | VALU | LDS |")
    print("|---|---|---|---|---|---|---|---|")
    for k, L in sorted(by.items(), key=lambda kv: -sum(c["SQ_WAVE_CYCLES"] for c in kv[1])):
        wc = np.array([c["SQ_WAVE_CYCLES"] for c in L])
        work = wc > 0.5 * np.percentile(wc, 90)

        def med(key):
            return float(np.median(np.array([c[key] for c in L])[work]))
        W = med("SQ_WAVE_CYCLES")
        print(f"| {k} | {len(L)} ({int(work.sum())}) | {W / med('SQ_BUSY_CU_CYCLES'):.1f} | "
              f"{med('SQ_WAIT_ANY') / W:.2f} | {med('SQ_ACTIVE_INST_ANY') / W:.2f} | "
              f"{med('SQ_ACTIVE_INST_VMEM') / W:.2f} | {med('SQ_ACTIVE_INST_VALU') / W:.2f} | "
              f"{med('SQ_ACTIVE_INST_LDS') / W:.2f} |")


def calibrate_copy():
    """Three device-to-device copies of 1 GiB (the HIP runtime's copy kernel: reads 1 GiB,
    writes 1 GiB), the yardstick for the FETCH_SIZE / WRITE_SIZE counters.  Plain HIP calls
    through ctypes, so the profiled process loads no other GPU library."""
    import ctypes
    try:
        hip = ctypes.CDLL("libamdhip64.so")
    except OSError:
        hip = ctypes.CDLL("/opt/rocm/lib/libamdhip64.so")
    n = 1 << 30
    a, b = ctypes.c_void_p(), ctypes.c_void_p()
    for ptr in (a, b):
        if hip.hipMalloc(ctypes.byref(ptr), ctypes.c_size_t(n)) != 0:
            raise RuntimeError("hipMalloc failed")
    if hip.hipMemset(a, 0, ctypes.c_size_t(n)) != 0:
        raise RuntimeError("hipMemset failed")
    for _ in range(3):
        if hip.hipMemcpy(b, a, ctypes.c_size_t(n), 3) != 0:   # hipMemcpyDeviceToDevice
            raise RuntimeError("hipMemcpy failed")
    hip.hipDeviceSynchronize()
    hip.hipFree(a)
    hip.hipFree(b)
    print(f"# calibration: 3 device-to-device copies of {n} bytes", file=sys.stderr, flush=True)


def aa_pass_bytes(npass, depth, mixed):
    """Algorithmic bytes per cell of the Anderson passes of one step (k_picard_next after every
    Picard iteration but the last).  Pass j combines min(j, depth) earlier passes; its first sweep
    reads x, psi_m and the ring's f and writes f, y, its second reads the ring's y and Ks and
    writes psi_m, theta, K, C (+ K32)."""
    total = 0
    for j in range(npass):
        nc = min(j, depth)
        total += 8 * (2 + nc + 2) + 8 * (nc + 1) + 8 * 4 + (4 if mixed else 0)
    return total


def mg_single_block_only(nx, ny, threads=1024):
    """True when every level of the overland multigrid fits the single-block kernel (the
    surface has no tiled level), as the library decides it."""
    total = 0   # the coarser levels' cells: one thread for each, down to the exact level
    while nx * ny > 64:
        nx, ny = (nx + 1) // 2, (ny + 1) // 2
        total += nx * ny
    return total <= threads


def counted_bytes(stats, n3, n2, mixed, olf_mg=True, one_kernel=False, column=False, aa_depth=0,
                  olf_cg1=False):
    """Algorithmic HBM bytes of the steps (per-kernel byte model of the solver)."""
    w = 4 if mixed else 8
    # overland CG iteration per surface cell: SpMV 6 and update 7 arrays; with the multigrid,
    # one V-cycle more: level 0 down (read b, d, we, wn; write x, 1/4 coarse b) and up (read
    # b, d, we, wn, x, 1/4 coarse y; write y), x 4/3 for the coarser levels.  Single-reduction
    # form (olf_cg1): no SpMV; the update inside the first down kernel reads w, s, r, z, p, x and
    # writes s, r, p, x (10 arrays), the down kernel then reads d, we, wn (b is the updated r)
    # and the up kernel also writes w = A z
    if olf_mg and olf_cg1:
        olf_iter = 10 * 8 + int(round((3 + 1.25 + 5.25 + 2) * 8 * 4 / 3))
    else:
        olf_iter = 13 * 8 + (int(round((4 + 1.25 + 5.25 + 1) * 8 * 4 / 3)) if olf_mg else 0)
    total = 0.0
    for s in stats:
        P, I, R, Io = s["picard_iters"], s["lin_iters"], s["refine_sweeps"], s["olf_iters"]
        # read x, psi_m, Ks; write theta, K, C, psi_m.  With the Anderson update the pass after a
        # solve reads x, psi_m for the increment alone (16 B); theta, K, C of the final x (read
        # x, Ks; write theta, K, C: 40 B) follow once per step, those of the other iterates come
        # with the Anderson passes
        vg = (16 if aa_depth else 56 + (4 if mixed else 0))
        asm = 80 if not mixed else 84                  # read 7 fields; write D, b, r (or D, b, D32, r32, d32)
        if column:
            # SpMV (read z, p, K, D; write p, q) + column kernel (read x, p, q, r, K, D; write
            # x, r, z) per iteration, a column start-up (read r, K, D; write z) per solve; a
            # reliable update (x += d, then the FP64 residual with the next segment's z in one
            # kernel) is the R * 64 below
            krylov = I * 15 * w + P * 4 * w
        elif one_kernel:
            # one launch per iteration: read r, D, p, K, x; write r, p, x (8 arrays), plus a
            # start-up pass per segment (read r, D, K, p: 4 arrays)
            krylov = I * 8 * w + (P + R) * 4 * w
        else:
            krylov = I * 13 * w
        per_cell = P * (vg + asm) + krylov + R * 64 + 48
        if aa_depth:
            # the last pass (converged, or at the iteration limit) evaluates theta, K, C of x instead
            per_cell += 40 + (4 if mixed else 0) + aa_pass_bytes(P - 1, aa_depth, mixed)
        per_surf = olf_iter * Io + 200                 # overland CG + surface/overland passes
        total += n3 * per_cell + n2 * per_surf
    return total


def run_timed(model, w, steps, marks=()):
    """Run `steps` steps; return (stats, seconds, snapshots at the requested step indices)."""
    snaps = {}
    bounds = sorted({0, steps, *[m for m in marks if 0 < m < steps]})
    stats = []
    elapsed = 0.0
    for a, b in zip(bounds[:-1], bounds[1:]):
        if a in marks:
            snaps[a] = (model.download("PSI"), model.download("PONDING"))
        t0 = time.perf_counter()
        stats += w.run(model, b - a, start=a)       # every library call returns synchronised
        elapsed += time.perf_counter() - t0
    if steps in marks:
        snaps[steps] = (model.download("PSI"), model.download("PONDING"))
    return stats, elapsed, snaps


def main():
    args = parse()
    if args.trace_summary:
        return trace_summary(args.trace_summary)
    if args.pmc_summary:
        return pmc_summary(*args.pmc_summary)
    if args.sq_summary:
        return sq_summary(args.sq_summary)
    if args.gpus != 1:
        print(json.dumps({"error": "bench.py measures one GPU; multi-GPU runs are not "
                                   "implemented (the domain decomposition is a design note)"}))
        sys.exit(2)
    import dhara_amd
    from dhara_amd import _abi, inputs

    dhara_amd.load_hip_library()            # raises without the HIP build; no fallback
    dev = dhara_amd.device_info()
    print(f"# device: {dev}", file=sys.stderr, flush=True)
    if args.calibrate_copy:
        calibrate_copy()
    if args.workload == "ensemble":
        return bench_ensemble(args, dev)
    K, W = args.steps, args.warmup
    nx, ny, nz = args.nx, args.ny, args.nz
    n3, n2 = nx * ny * nz, nx * ny

    def cp(p):
        return _abi.Params.from_buffer_copy(p)

    w64 = inputs.c2_coupled(nx=nx, ny=ny, nz=nz)
    w32 = inputs.c3_coupled_mixed(nx=nx, ny=ny, nz=nz)
    column = args.precond == "column"
    one_kernel = args.krylov == "one" and not column
    for w_ in (w64, w32):
        w_.params.krylov = _abi.KRYLOV_ONE_KERNEL if args.krylov == "one" else _abi.KRYLOV_TWO_KERNEL
        w_.params.precond = _abi.PRECOND_COLUMN if column else _abi.PRECOND_JACOBI
    if args.refine_max is not None:
        w32.params.refine_maxiter = args.refine_max
    if args.inner_tol is not None:
        w32.params.inner_tol = args.inner_tol
    if args.mixed_lin_tol is not None:
        w32.params.lin_tol = args.mixed_lin_tol
    runs = {}
    order = [("fp64", w64), ("mixed", w32)]
    if args.only != "both":
        order = [o for o in order if o[0] == args.only]
    cpu_start = min(args.cpu_start, max(K - args.cpu_steps, 0))
    cpu_marks = (cpu_start, cpu_start + args.cpu_steps)
    tiles = {}
    for name, w in order:
        # warm-up on a throw-away context, then the tile autotuner on its operator; the tuned
        # shape goes to the library's process-wide table, which the timed context reads
        pinned = {8: args.tile_f64, 4: args.tile_f32}
        m = dhara_amd.FlowModel(w.grid, cp(w.params))
        w.apply(m)
        w.run(m, max(W, 1))
        tune_us = m.autotune() if not any(pinned.values()) else (0.0, 0.0)
        m.close()
        m = dhara_amd.FlowModel(w.grid, cp(w.params))
        for eb, spec in pinned.items():
            if spec:
                m.set_tile(eb, *[int(v) for v in spec.split(",")])
        m_tile_fp64 = m.get_krylov_tile(8) if one_kernel else m.get_tile(8)
        m_tile_fp32 = m.get_krylov_tile(4) if one_kernel else m.get_tile(4)
        if one_kernel:
            tiles[name] = {"fp64": m.get_krylov_tile(8), "fp32": m.get_krylov_tile(4), "tune_us": tune_us,
                           "kernel": "k_cg1 (tx, ty, planes per tile, grid cap)"}
        else:
            tiles[name] = {"fp64": m.get_tile(8), "fp32": m.get_tile(4), "tune_us": tune_us,
                           "kernel": "k_pcg3_spmv_tiled (tx, ty, planes per block)"
                                     + ("; column solve: one thread per column" if column else "")}
        w.apply(m)
        print(f"# {name}: {K} steps", file=sys.stderr, flush=True)
        stats, secs, snaps = run_timed(m, w, K, marks=(cpu_marks + (K,)) if name == "fp64" else (K,))
        # kernel timestamps (an event pair per Krylov launch) only outside the timed region
        m.profile(True)
        w.run(m, args.prof_steps, start=K)
        prof = m.profile_read()
        m.profile(False)
        psi = m.download("PSI")
        h = m.download("PONDING")
        m.close()
        runs[name] = dict(stats=stats, secs=secs, snaps=snaps, prof=prof, psi=psi, h=h,
                          tile=(m_tile_fp32 if name == "mixed" else m_tile_fp64))
        print(f"# {name}: {secs:.3f} s, {n3 * K / secs:.4e} cell-steps/s, picard "
              f"{sum(s['picard_iters'] for s in stats)}, krylov {sum(s['lin_iters'] for s in stats)}",
              file=sys.stderr, flush=True)

    # the plain method (FP64 end to end, Jacobi-PCG, one-kernel form) on the same workload, for
    # the speed-up of the fast path over it
    # and the mixed-precision form of the same Jacobi-PCG (the survey's wording of the mixed
    # configuration), so that precision and preconditioner can be told apart
    plain = mixed_jacobi = None
    if column and not args.no_plain and args.only == "both":
        def jacobi_run(wj, label):
            wj.params.krylov = _abi.KRYLOV_ONE_KERNEL
            wj.params.precond = _abi.PRECOND_JACOBI
            m = dhara_amd.FlowModel(wj.grid, cp(wj.params))
            wj.apply(m)
            wj.run(m, max(W, 1))
            m.autotune()
            m.close()
            m = dhara_amd.FlowModel(wj.grid, cp(wj.params))
            wj.apply(m)
            print(f"# {label}: {K} steps", file=sys.stderr, flush=True)
            st_j, secs_j, snaps_j = run_timed(m, wj, K, marks=(K,))
            m.close()
            res = {"cell_steps_per_s": n3 * K / secs_j, "seconds": secs_j,
                   "picard_iters": sum(s_["picard_iters"] for s_ in st_j),
                   "krylov_iters": sum(s_["lin_iters"] for s_ in st_j),
                   "picard_unconverged_steps": sum(1 for s_ in st_j if not s_["picard_converged"])}
            print(f"# {label}: {secs_j:.3f} s, {res['cell_steps_per_s']:.4e} cell-steps/s", file=sys.stderr, flush=True)
            return res, snaps_j[K][0]
        plain, psi_pj = jacobi_run(inputs.c2_coupled(nx=nx, ny=ny, nz=nz), "plain fp64 (Jacobi)")
        plain["solver"] = "FP64 Jacobi-PCG, one-kernel form, tuned tile"
        mixed_jacobi, psi_mj = jacobi_run(inputs.c3_coupled_mixed(nx=nx, ny=ny, nz=nz), "mixed (Jacobi)")
        mixed_jacobi["solver"] = "FP32 Jacobi-PCG with FP64 reliable updates, one-kernel form, tuned tile"
        mixed_jacobi["head_error_vs_plain_fp64_max_m"] = float(np.max(np.abs(psi_mj - psi_pj)))
    head = "mixed" if "mixed" in runs else "fp64"
    r = runs[head]
    value = n3 * K / r["secs"]
    out = {
        "metric": METRIC, "value": value, "unit": "cell-steps/s", "n_gpus": 1, "steps": K,
        "warmup": W, "ms_per_step": 1e3 * r["secs"] / K, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None,
        "dtype": "f32+f64" if head == "mixed" else "f64",
        "data": "synthetic (seeded GRF topography and log-normal Ks; no external data)",
        "config": {"workload": f"coupled {nx}x{ny}x{nz} (surface {nx}x{ny}), 20 mm/h rain 3600 s + "
                               f"3600 s recession, dt 30 s; {head} run timed over steps 0..{K - 1}",
                   "precision": head, "device": dev, "precond": args.precond,
                   "krylov": "two (column-solve kernel)" if column else args.krylov, "tiles": tiles,
                   "mixed_solver": {"refine_maxiter": w32.params.refine_maxiter, "inner_tol": w32.params.inner_tol,
                                    "lin_tol": w32.params.lin_tol},
                   "fp64_solver": {"lin_tol": w64.params.lin_tol}},
    }
    for name, rr in runs.items():
        st = rr["stats"]
        out[name] = {
            "cell_steps_per_s": n3 * K / rr["secs"], "seconds": rr["secs"],
            "picard_iters": sum(s["picard_iters"] for s in st),
            "krylov_iters": sum(s["lin_iters"] for s in st),
            "refine_sweeps": sum(s["refine_sweeps"] for s in st),
            "overland_iters": sum(s["olf_iters"] for s in st),
            "picard_unconverged_steps": sum(1 for s in st if not s["picard_converged"]),
            "max_mb_rel_all_steps": max(s["mb_rel"] for s in st),
            # the balance of the whole window: |sum(storage change - boundary inflow)| over the
            # sum of |storage change| (m^3), i.e. the subsurface water the steps created or lost
            "cumulative_mb_rel": abs(sum(s["storage_change"] - s["boundary_inflow"] for s in st)) /
            max(sum(abs(s["storage_change"]) for s in st), 1e-300),
            "counted_hbm_bytes": counted_bytes(st, n3, n2, name == "mixed", one_kernel=one_kernel, column=column,
                                               aa_depth=w64.params.picard_accel,
                                               olf_cg1=not mg_single_block_only(args.nx, args.ny)),
        }
        out[name]["step_hbm_frac"] = out[name]["counted_hbm_bytes"] / (rr["secs"] * HBM_PEAK)
    out["config"]["picard"] = {"tol_m": w64.params.picard_tol, "maxiter": w64.params.picard_maxiter,
                               "anderson_depth": w64.params.picard_accel, "am": w64.params.am,
                               "initial_water_table_m": inputs.C2_WATER_TABLE}
    if "fp64" in runs and "mixed" in runs:
        # heads at the end of the timed window (step K) of both runs
        p64, h64 = runs["fp64"]["snaps"][K]
        p32, h32 = runs["mixed"]["snaps"][K]
        d = p32 - p64
        err = float(np.max(np.abs(d)))
        out["mixed_over_fp64"] = runs["fp64"]["secs"] / runs["mixed"]["secs"]
        out["head_error_vs_fp64"] = {"max_m": err, "rms_m": float(np.sqrt(np.mean(d * d))),
                                     "ponding_max_m": float(np.max(np.abs(h32 - h64))),
                                     "after_step": K, "target_m": 1e-6, "within_target": err <= 1e-6}
        out["config"]["head_error_target"] = ("met: mixed within 1e-6 m of FP64 after the timed steps"
                                              if err <= 1e-6 else
                                              f"MISSED: mixed {err:.2e} m from FP64 after the timed steps")
    if plain is not None:
        out["plain_fp64_jacobi"] = plain
        out["mixed_jacobi"] = mixed_jacobi
        out["mixed_jacobi_over_plain_fp64"] = plain["seconds"] / mixed_jacobi["seconds"]
        if "mixed" in runs:
            out["mixed_over_plain_fp64"] = plain["seconds"] / runs["mixed"]["secs"]
    # roofline of the dominant kernel, from the library's HIP-event timing
    pr = r["prof"]
    kern = []
    names = ((("pcg3_spmv_z" if column else "cg1" if one_kernel else "pcg3_spmv"), "spmv"),
             (("line" if column else "pcg_update"), "update"))
    for kname, key in names:
        nl = pr[f"{key}_launches"]
        if nl:
            avg = pr[f"{key}_ms"] / nl * 1e-3
            kern.append((pr[f"{key}_ms"], kname, avg, pr[f"{key}_bytes"], nl))
    if pr["aa_launches"]:   # the Anderson Picard pass (FP64; bytes vary with its ring: the mean)
        nl = pr["aa_launches"]
        kern.append((pr["aa_ms"], "picard_next", pr["aa_ms"] / nl * 1e-3, pr["aa_bytes"] / nl, nl))
    if kern:
        kern.sort(reverse=True)
        tot, kname, avg, byts, nl = kern[0]
        kprec = "f32" if pr["elem_bytes"] == 4 else "f64"
        prec = "f64" if kname == "picard_next" else kprec
        # measured HBM bytes per launch (rocprof PMC, copy-calibrated) for the tile in use, if the
        # profile holds that tile
        traffic = None
        tpath = os.path.join(ROOT, "profiles", "traffic.json")
        if os.path.exists(tpath):
            try:
                entry = json.load(open(tpath)).get(f"k_{kname}<{prec}>")
                tile_now = list(r["tile"]) if r.get("tile") is not None else None
                if isinstance(entry, dict) and ("tile" not in entry or entry["tile"] == tile_now):
                    traffic = entry["bytes_per_launch"]
            except Exception:
                traffic = None
        out["roofline"] = {"bound": "hbm", "kernel": f"k_{kname}<{prec}>",
                           "tile": None if kname == "picard_next" else r.get("tile"),
                           "achieved": byts / avg / 1e9,
                           "peak": HBM_PEAK / 1e9, "unit": "GB/s", "frac": byts / avg / HBM_PEAK,
                           "traffic": traffic, "avg_us": avg * 1e6, "launches": nl,
                           "bytes_per_launch": byts}
        out["roofline"]["total_ms"] = tot
        out["roofline_other_kernels"] = [
            {"kernel": f"k_{k[1]}<{'f64' if k[1] == 'picard_next' else kprec}>", "achieved": k[3] / k[2] / 1e9,
             "frac": k[3] / k[2] / HBM_PEAK, "avg_us": k[2] * 1e6, "launches": k[4], "total_ms": k[0]}
            for k in kern[1:]]
    # CPU baseline: oracle on a bounded window, from the GPU FP64 state
    if not args.no_cpu and "fp64" in runs and cpu_start in runs["fp64"]["snaps"]:
        from oracle import oracle
        threads = oracle.set_threads(0)
        om = oracle.OracleModel(w64.grid, cp(w64.params),
                                lin_solver=oracle.LIN_PCG_LINE if column else oracle.LIN_PCG_JACOBI)
        om.upload_many(w64.fields)
        psi0, h0 = runs["fp64"]["snaps"][cpu_start]
        om.upload("PSI", psi0)
        om.upload("PONDING", h0)
        om.init_state(_abi.INIT_FROM_PSI)
        print(f"# cpu oracle: steps {cpu_start}..{cpu_start + args.cpu_steps - 1} on {threads} threads",
              file=sys.stderr, flush=True)
        t0 = time.perf_counter()
        w64.run(om, args.cpu_steps, start=cpu_start)
        cs = time.perf_counter() - t0
        gpu_win = sum(s["wall_ms"] for s in runs["fp64"]["stats"][cpu_start:cpu_start + args.cpu_steps]) * 1e-3
        psi_c = om.download("PSI")
        psi_g = runs["fp64"]["snaps"].get(cpu_start + args.cpu_steps, (None,))[0]
        out["cpu_baseline"] = {
            "value": n3 * args.cpu_steps / cs, "unit": "cell-steps/s", "cores": threads,
            "kind": "port",
            "sample": f"oracle FP64 (C++/OpenMP, {'column' if column else 'Jacobi'}-preconditioned CG) on steps "
                      f"{cpu_start}..{cpu_start + args.cpu_steps - 1} of the "
                      f"{nx}x{ny}x{nz} coupled workload, started from the GPU FP64 state",
            "seconds": cs, "gpu_fp64_same_steps_s": gpu_win,
            "gpu_fp64_speedup_same_steps": cs / gpu_win if gpu_win > 0 else None,
            "max_head_diff_vs_gpu_fp64_m": float(np.max(np.abs(psi_c - psi_g))) if psi_g is not None else None,
        }
        om.close()
        if args.cpu_1thread_steps > 0:
            # the same window's first steps again on one host thread
            k1 = min(args.cpu_1thread_steps, args.cpu_steps)
            oracle.set_threads(1)
            om = oracle.OracleModel(w64.grid, cp(w64.params),
                                    lin_solver=oracle.LIN_PCG_LINE if column else oracle.LIN_PCG_JACOBI)
            om.upload_many(w64.fields)
            om.upload("PSI", psi0)
            om.upload("PONDING", h0)
            om.init_state(_abi.INIT_FROM_PSI)
            print(f"# cpu oracle: step {cpu_start}..{cpu_start + k1 - 1} on 1 thread", file=sys.stderr, flush=True)
            t0 = time.perf_counter()
            w64.run(om, k1, start=cpu_start)
            c1s = time.perf_counter() - t0
            om.close()
            oracle.set_threads(threads)
            gpu1 = sum(s["wall_ms"] for s in runs["fp64"]["stats"][cpu_start:cpu_start + k1]) * 1e-3
            out["cpu_baseline_1thread"] = {"value": n3 * k1 / c1s, "unit": "cell-steps/s", "cores": 1,
                                           "kind": "port", "seconds": c1s,
                                           "sample": f"steps {cpu_start}..{cpu_start + k1 - 1} of the same window",
                                           "gpu_fp64_speedup_same_steps": c1s / gpu1 if gpu1 > 0 else None}
    if not args.no_c1:
        out["c1"] = bench_c1(args, column)
    print(json.dumps(out))


def bench_c1(args, column):
    """C1 (32x32x20 homogeneous loam, 100 steps of 60 s) in full: the GPU FP64 path and the CPU
    oracle on all host threads and on one, the same solver, and the largest head difference."""
    import dhara_amd
    from dhara_amd import _abi, inputs
    from oracle import oracle
    w = inputs.c1_column()
    p = _abi.Params.from_buffer_copy(w.params)
    p.precond = _abi.PRECOND_COLUMN if column else _abi.PRECOND_JACOBI
    n3 = w.ncells
    out = {"workload": "C1 32x32x20, 100 steps, FP64, reference Picard update, Picard 1e-6 m, PCG 1e-12"}
    gm = dhara_amd.FlowModel(w.grid, _abi.Params.from_buffer_copy(p))
    w.apply(gm)
    gm.step(1)                                   # warm-up (kernel loading), then a fresh state
    gm.close()
    gm = dhara_amd.FlowModel(w.grid, _abi.Params.from_buffer_copy(p))
    w.apply(gm)
    t0 = time.perf_counter()
    st = gm.step(w.nsteps)
    gs = time.perf_counter() - t0
    psi_g = gm.download("PSI")
    gm.close()
    out["gpu"] = {"cell_steps_per_s": n3 * w.nsteps / gs, "seconds": gs,
                  "picard_iters": sum(s["picard_iters"] for s in st),
                  "max_mb_rel": max(s["mb_rel"] for s in st),
                  "unconverged_steps": sum(1 for s in st if not s["picard_converged"])}
    ls = oracle.LIN_PCG_LINE if column else oracle.LIN_PCG_JACOBI
    threads = oracle.set_threads(0)
    for key, nt in (("cpu", threads), ("cpu_1thread", 1)):
        oracle.set_threads(nt)
        om = oracle.OracleModel(w.grid, _abi.Params.from_buffer_copy(p), lin_solver=ls)
        w.apply(om)
        t0 = time.perf_counter()
        om.step(w.nsteps)
        cs = time.perf_counter() - t0
        out[key] = {"cell_steps_per_s": n3 * w.nsteps / cs, "seconds": cs, "cores": nt,
                    "max_head_diff_vs_gpu_m": float(np.max(np.abs(om.download("PSI") - psi_g)))}
        om.close()
    oracle.set_threads(threads)
    print(f"# C1: GPU {gs:.3f} s, CPU {out['cpu']['seconds']:.3f} s ({threads} threads), "
          f"{out['cpu_1thread']['seconds']:.3f} s (1 thread)", file=sys.stderr, flush=True)
    return out


def bench_ensemble(args, dev):
    """The batched ensemble: members with nx, ny ~ U{32..128}, nz ~ U{10..40}, their own seeded
    log-normal Ks (sigma ~ U[0.5, 1.5]), per-cell alpha ~ U[2,5], n ~ U[1.3,1.8], rain ~ U[5,50]
    mm/h, dt = 30 s, stepped together in mixed precision; the same members in FP64 (an FP64
    ensemble equals each member stepped alone, bit for bit) give the per-member head error."""
    import dhara_amd
    from dhara_amd import _abi, inputs
    specs = inputs.c5_instances()[:args.members]
    K = args.steps if args.steps != 240 else 200
    ws = [inputs.c5_member(sp) for sp in specs]
    ncell = sum(w.ncells for w in ws)

    column = args.precond == "column"

    def build(prec):
        ms = []
        for w in ws:
            p = _abi.Params.from_buffer_copy(w.params)
            p.precision = prec
            p.precond = _abi.PRECOND_COLUMN if column else _abi.PRECOND_JACOBI
            if args.inner_tol is not None:
                p.inner_tol = args.inner_tol
            m = dhara_amd.FlowModel(w.grid, p)
            w.apply(m)
            ms.append(m)
        return ms

    res = {}
    for name, prec in (("mixed", _abi.MIXED), ("fp64", _abi.FP64)):
        if args.only not in ("both", name):
            continue
        ms = build(prec)
        ens = dhara_amd.Ensemble(ms)
        if args.no_graph:
            ens.set_graph(False)
        if column:   # the column form's kernels are untiled: nothing to tune
            tune_us, div = 0.0, 0
            print(f"# ensemble {name}: {len(ms)} members, {ncell:.4e} cells, {K} steps; column-preconditioned PCG",
                  file=sys.stderr, flush=True)
        else:
            tune_us, div = ens.autotune()   # planes per tile of the batched one-kernel PCG (untimed)
            floor_us = ncell * 8 * (4 if prec == _abi.MIXED else 8) / 8e12 * 1e6   # 8 arrays at 8 TB/s
            print(f"# ensemble {name}: {len(ms)} members, {ncell:.4e} cells, {K} steps; tiles 32x8 x ceil(nz/{div}) "
                  f"({tune_us:.0f} us per batched iteration, HBM floor {floor_us:.0f} us)", file=sys.stderr,
                  flush=True)
        t0 = time.perf_counter()
        st = []
        for k in range(0, K, 20):
            st += ens.step(min(20, K - k))
            print(f"#   step {k + 20}: {time.perf_counter() - t0:.1f} s", file=sys.stderr, flush=True)
        secs = time.perf_counter() - t0
        res[name] = dict(secs=secs, stats=st, psi=[m.download("PSI") for m in ms], div=div, tune_us=tune_us)
        ens.close()
        for m in ms:
            m.close()
    if len(res) < 2:   # one precision only (profiling runs): its time and counts
        (name, r), = res.items()
        flat = [x for row in r["stats"] for x in row]
        print(json.dumps({"workload": "ensemble", "precision": name, "members": len(ws), "cells": ncell, "steps": K,
                          "seconds": r["secs"], "cell_steps_per_s": ncell * K / r["secs"],
                          "picard_iters": sum(x["picard_iters"] for x in flat),
                          "krylov_iters": sum(x["lin_iters"] for x in flat),
                          "refine_sweeps": sum(x["refine_sweeps"] for x in flat),
                          "olf_iters": sum(x["olf_iters"] for x in flat)}))
        return
    err = np.array([np.max(np.abs(a - b)) for a, b in zip(res["mixed"]["psi"], res["fp64"]["psi"])])
    r = res["mixed"]
    flat = [x for row in r["stats"] for x in row]
    out = {
        "metric": "aggregate cell-steps/s of the batched ensemble (mixed precision)", "value": ncell * K / r["secs"],
        "unit": "cell-steps/s", "n_gpus": 1, "steps": K, "warmup": 0, "ms_per_step": 1e3 * r["secs"] / K,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32+f64",
        "data": "synthetic (seeded GRF Ks and topography per member, uniform draws of alpha, n, rain)",
        "config": {"workload": f"batched ensemble of {len(ws)} members (nx, ny in 32..128, nz in 10..40), "
                               f"{ncell} cells in total, dt 30 s, {K} steps, one launch per kernel for all members, "
                               f"Krylov batches replayed from a captured hipGraph, every member's overland "
                               f"multigrid CG in one launch (a workgroup per member)", "device": dev,
                   "precond": args.precond,
                   "krylov_tiles": ({n_: "untiled SpMV + one thread per column (column-preconditioned PCG)"
                                     for n_ in res} if column else
                                    {n_: f"32x8 columns x ceil(nz/{res[n_]['div']}) planes, "
                                         f"{res[n_]['tune_us']:.0f} us per batched iteration (ensemble autotuner)"
                                     for n_ in res})},
        "fp64": {"cell_steps_per_s": ncell * K / res["fp64"]["secs"], "seconds": res["fp64"]["secs"]},
        "mixed": {"seconds": r["secs"], "picard_iters": sum(x["picard_iters"] for x in flat),
                  "krylov_iters": sum(x["lin_iters"] for x in flat),
                  "unconverged_member_steps": sum(1 for x in flat if not x["picard_converged"])},
        "head_error_vs_fp64_per_member": {"max_m": float(err.max()), "median_m": float(np.median(err)),
                                          "members_within_1e-6_m": int(np.sum(err <= 1e-6)),
                                          "members": len(ws)},
    }
    print(json.dumps(out))


if __name__ == "__main__":
    main()
