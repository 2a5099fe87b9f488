#!/usr/bin/env python3
"""Benchmark of the headline workload on one MI355X.

Workload: 3D 7-point Poisson on a 128^3 grid (n = 2,097,152, nnz = 14,581,760),
b = A x*, x* ~ U(-1, 1) from the library's seeded stream (seed 0), x0 = 0, CG to
true relative residual 1e-10.  One step = one full solve from x0 = 0 with b and
x resident in HBM (device buffers owned by torch, passed to mf_solve_device).

Reported: time to tolerance of the per-tile mixed-precision solve (the value),
the same persistent kernel run FP64-only, their ratio, the standalone tiled
SpMV kernel's bandwidth, the roofline of the dominant kernel (the persistent
CG kernel: one SpMV at its algorithmic bytes per unit), the batched solve of
512 systems x 8 right-hand sides, the oracle's tile-SpMV CG and the restated
PETSc CG timed on the host cores, and the same records for the other single
system workloads: the 256^2 Laplacian CG, the 96^3 convection-diffusion
BiCGSTAB and the random SPD (n = 1M) CG.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu] [--no-batched] [--no-configs]
    (profiling aids: --only-batched [--batched-no-tune], --only-bicgstab, --only-config NAME, --calib)
"""
import argparse
import json
import os
import statistics
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "time to rel. residual 1e-10 (ms), SpMV HBM GB/s; mixed vs FP64-only speedup"
HBM_PEAK = 8.0e12
TOL = 1e-10


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def host_cpu():
    """The host the CPU baselines run on: logical CPUs, the CPUs this process
    may run on, the model name, OMP_NUM_THREADS, and the thread count used
    (OMP_NUM_THREADS when set -- a GPU box sets it to its CPU share -- else
    every CPU of the affinity mask)."""
    model = None
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    aff = len(os.sched_getaffinity(0))
    omp = os.environ.get("OMP_NUM_THREADS")
    threads = int(omp) if omp and omp.isdigit() and int(omp) > 0 else aff
    return {"nproc": os.cpu_count(), "affinity_cpus": aff, "model": model, "OMP_NUM_THREADS": omp,
            "threads": threads}


def _oracle():
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    from orc import Oracle
    return Oracle()


def cpu_baseline(rp, ci, va, b, gpu_iters, gpu_x=None):
    """The oracle's tile-SpMV CG (FP64, OpenMP over the host cores) run to the
    same tolerance on the same system; gpu_x maps a label to a GPU solution,
    whose relative error against the oracle's solution is reported."""
    O = _oracle()
    n = len(b)
    host = host_cpu()
    cores = host["threads"]
    T = O.tiles(16, n, n, rp, ci, va)
    t0 = time.perf_counter()
    x, rep = O.cg(rp, ci, va, b, TOL, 20000, tiles=T, nthreads=cores)
    dt = (time.perf_counter() - t0) * 1e3
    # the restated PETSc KSPCG (CSR SpMV; its stopping test is the updated
    # residual, so its true relres is reported beside it)
    t0 = time.perf_counter()
    _, prep = O.petsc_cg(rp, ci, va, b, TOL, 20000, nthreads=cores)
    dp = (time.perf_counter() - t0) * 1e3
    return {
        "value": round(dt, 3), "unit": "ms", "cores": cores, "kind": "port",
        "sample": f"full solve: oracle tile-SpMV CG (FP64, {cores} OpenMP threads) to true relres "
                  f"{TOL:g} on the same 128^3 system, {rep.iterations} iterations "
                  f"(GPU FP64: {gpu_iters}), relres {rep.relres_true:.2e}",
        "iterations": rep.iterations,
        "petsc_cg": {"ms": round(dp, 3), "iterations": prep.iterations, "relres_true": prep.relres_true,
                     "kind": "port", "cores": cores},
        "host": host,
        "gpu_err_vs_oracle_x": {k: float(np.linalg.norm(v - x) / np.linalg.norm(x))
                                for k, v in (gpu_x or {}).items()},
    }


def calibration_copy(torch):
    """Three device copies of 512 MiB (known bytes) for the PMC byte counters."""
    src = torch.ones(64 << 20, dtype=torch.float64, device="cuda")
    dst = torch.empty_like(src)
    for _ in range(3):
        dst.copy_(src)
    torch.cuda.synchronize()
    log(f"calibration copy: {src.numel() * 8} bytes read and written per launch, 3 launches")
    del src, dst


def batched_run(mf, nsys=512, nrhs=8, tune=True):
    """512 independent SPD systems, n log-uniform in [1k, 64k] (library
    stream, seed 0), alternating 2D 5-point and 3D 7-point stencils with
    lognormal(sigma = 1.5) cell coefficients (grids padded up to n), 8
    right-hand sides N(0, 1) each; one graph-captured persistent launch,
    workgroups and tile size picked by the autotuner."""
    t0 = time.perf_counter()
    u = mf.gen_uniform(0, nsys, np.log(1000.0), np.log(64000.0))
    sizes = np.exp(u).astype(int)
    systems = [mf.gen_stencil_lognormal(2 if i % 2 == 0 else 3, int(sizes[i]), 1.5, 1000 + i) for i in range(nsys)]
    rng = np.random.default_rng(0)
    b = [rng.standard_normal((nrhs, len(s[0]) - 1)) for s in systems]
    # mixed precision requested: per-tile classes (lossless at first); the
    # tuner also tries FP32- and FP16-rounded tiles and keeps the fastest
    # configuration in which every column converges
    bt = mf.Batch(systems, nrhs=nrhs, tol=TOL, precision=mf.MF_MIXED, tau=0.0, rr_factor=1e-2)
    t1 = time.perf_counter()
    if tune:
        bt.tune(b)
    t2 = time.perf_counter()
    info = bt.info()
    reps = []
    for _ in range(2):
        xs, it, rel, rep = bt.solve(b)
        if rep["status"] != 0 or rel.max() > TOL:
            raise RuntimeError(f"batched solve did not reach tolerance: {rep}")
        reps.append(rep["ms_solve"])
    ms = min(reps)
    n = np.array([len(s[0]) - 1 for s in systems], dtype=np.float64)
    # algorithmic bytes: each system's share (by rows) of the per-iteration
    # bytes (matrix once + 16 n per column) times its own iterations
    alg = float(np.sum(info["bytes_alg"] * n / n.sum() * it))
    bt.close()
    log(f"batched: {nsys} systems x {nrhs} rhs, setup {t1 - t0:.1f}s, tune {t2 - t1:.1f}s ({info['tuned']}), "
        f"solve {ms:.1f} ms, iterations max {it.max()} mean {it.mean():.0f}")
    return {"ms": round(ms, 2), "systems": nsys, "rhs_per_system": nrhs, "rows": int(n.sum()),
            "nnz": int(sum(len(s[1]) for s in systems)), "iterations_max": int(it.max()),
            "iterations_mean": round(float(it.mean()), 1), "relres_max": float(rel.max()),
            "B": info["B"], "workgroups": info["G"], "tuned": info["tuned"],
            "bytes_alg_total": alg, "GBps": round(alg / (ms * 1e-3) / 1e9, 1),
            "frac": round(alg / (ms * 1e-3) / HBM_PEAK, 4),
            "tile_precision": ("mixed tau=%g" % info["tau"]) if info["mixed"] else "fp64",
            "nnz_per_code": info["nnz_per_code"]}


def _roofline(iters, spmvs_per_iter, bytes_alg, ms):
    """One SpMV at its algorithmic bytes (B_alg = min(tile, CSR) bytes: values
    and indices, tile metadata, the gathered vector read once, y written once)
    is the unit; a solve runs iterations x SpMVs per iteration of them."""
    ach = iters * spmvs_per_iter * bytes_alg / (ms * 1e-3)
    return {"bound": "hbm", "achieved": round(ach / 1e9, 1), "peak": HBM_PEAK / 1e9, "unit": "GB/s",
            "frac": round(ach / HBM_PEAK, 4), "bytes_per_unit": bytes_alg,
            "units_per_launch": iters * spmvs_per_iter}


def _configs(mf):
    """The single-system workloads besides the headline, as generators:
    (label, workload text, method, builder -> (rp, ci, va, x*), variants)."""
    def laplace():
        rp, ci, va = mf.gen_laplace2d(256, 256)
        return rp, ci, va, np.ones(len(rp) - 1)

    def convdiff():
        rp, ci, va = mf.gen_convdiff3d(96, 10.0, 1.0, 0)
        return rp, ci, va, mf.gen_uniform(0, len(rp) - 1, -1.0, 1.0)

    def random_spd():
        rp, ci, va = mf.gen_random_spd(1000000, 2.0, 2, 2000, 0)
        return rp, ci, va, mf.gen_uniform(0, len(rp) - 1, -1.0, 1.0)

    return {
        "laplace256_cg": ("2D 5-point Laplacian 256^2, CG to true relres 1e-10, b = A 1", mf.MF_CG, laplace,
                          {"fp64": dict(precision=mf.MF_FP64),
                           "mixed": dict(precision=mf.MF_MIXED, tau=0.0, rr_factor=1e-2)}),
        "convdiff96_bicgstab": ("27-point convection-diffusion 96^3 (cell Peclet 10, lognormal(1) diffusion), "
                                "BiCGSTAB to true relres 1e-10, b = A x*, x* ~ U(-1,1) seed 0", mf.MF_BICGSTAB,
                                convdiff,
                                {"fp64": dict(precision=mf.MF_FP64),
                                 "fp32_tiles": dict(precision=mf.MF_MIXED, tau=2.0 ** -24, rr_factor=1e-2),
                                 "fp16_tiles": dict(precision=mf.MF_MIXED, tau=2.0 ** -11, rr_factor=1e-2),
                                 "e4m3_tiles": dict(precision=mf.MF_MIXED, tau=2.0 ** -4, rr_factor=1e-2)}),
        "random_spd_1m_cg": ("random SPD n = 1,000,000 (Zipf(2) row lengths in [2, 2000], B + B^T, diagonal "
                             "1.05 x row abs-sum), CG to true relres 1e-10, b = A x*, x* ~ U(-1,1) seed 0", mf.MF_CG,
                             random_spd,
                             {"fp64": dict(precision=mf.MF_FP64),
                              "mixed": dict(precision=mf.MF_MIXED, tau=2.0 ** -24, rr_factor=1e-2)}),
    }


def config_run(mf, torch, name, steps, warmup, cpu=True):
    """One of the other single-system workloads: every variant of the
    persistent solver (median time to tolerance over the steps, b and x in
    HBM), its roofline on one SpMV at B_alg, the vendor-library baseline, and
    the oracle's tile solver and the restated PETSc solver on the host cores
    (to tolerance, or capped for the random SPD system, whose CSR solve runs
    seconds per hundred iterations on the host)."""
    import scipy.sparse as sp
    text, method, build, variants = _configs(mf)[name]
    t0 = time.perf_counter()
    rp, ci, va, xs = build()
    n = len(rp) - 1
    b = sp.csr_matrix((va, ci, rp), shape=(n, n)) @ xs
    A = mf.Matrix(rp, ci, va)
    info = A.info()
    dev = torch.device("cuda:0")
    npad = info["tilem"] * info["B"]
    d_b = torch.zeros(npad, dtype=torch.float64, device=dev)
    d_b[:n] = torch.from_numpy(b).to(dev)
    d_x = torch.zeros(npad, dtype=torch.float64, device=dev)
    torch.cuda.synchronize()
    log(f"{name}: n={n} nnz={len(ci)} set up in {time.perf_counter() - t0:.1f}s")
    spmvs = 2 if method == mf.MF_BICGSTAB else 1
    out = {"workload": text, "n": n, "nnz": int(len(ci)), "method": "bicgstab" if spmvs == 2 else "cg",
           "unit_def": "one SpMV at B_alg = min(tile, CSR) algorithmic bytes", "spmvs_per_iteration": spmvs}
    k = steps if n * 20 < 30e6 else max(2, min(steps, 3))  # the random SPD solve takes ~0.2 s
    xsol = {}
    for label, opts in variants.items():
        if opts.get("precision") == mf.MF_MIXED:
            A.layout(opts["tau"])
        balg = A.info()["bytes_alg_mixed" if opts.get("precision") == mf.MF_MIXED else "bytes_alg_fp64"]
        o = dict(method=method, tol=TOL, **opts)
        for _ in range(warmup):
            A.solve_device(d_b.data_ptr(), d_x.data_ptr(), **o)
        reps = [A.solve_device(d_b.data_ptr(), d_x.data_ptr(), **o) for _ in range(k)]
        ok = all(r["status"] == 0 and r["relres_true"] <= TOL for r in reps)
        ms = statistics.median(r["ms_solve"] for r in reps)
        it = reps[0]["iterations"]
        x = d_x[:n].cpu().numpy()
        xsol[label] = x
        rec = {"ms": round(ms, 4), "iterations": it, "replacements": reps[0]["replacements"],
               "relres_true": reps[0]["relres_true"], "converged": ok,
               "err_vs_xstar": float(np.linalg.norm(x - xs) / np.linalg.norm(xs)),
               "grid": reps[0]["grid"], "reordered": reps[0]["reordered"], "sync_deps": reps[0]["sync_deps"],
               "nnz_per_code": A.info()["nnz_per_code"] if opts.get("precision") == mf.MF_MIXED else None,
               "streamed": reps[0]["streamed"], "fallback": reps[0]["fallback"],
               "split_rows": reps[0]["split_rows"],
               "pattern_slabs": A.info()["pattern_slabs_mixed" if opts.get("precision") == mf.MF_MIXED
                                         else "pattern_slabs_fp64"],
               "roofline": _roofline(it, spmvs, balg, ms)}
        out[label] = rec
        log(f"{name} {label}: {ms:.3f} ms, {it} it, converged {ok}, roofline {rec['roofline']['frac']}")
    for label in variants:
        if label != "fp64" and out[label]["converged"]:
            out[f"speedup_{label}_vs_fp64"] = round(out["fp64"]["ms"] / out[label]["ms"], 3)
    v = A.vendor_solve_device(d_b.data_ptr(), d_x.data_ptr(), method=method, tol=TOL)
    out["vendor_baseline"] = {"ms": round(v["ms_solve"], 3), "iterations": v["iterations"],
                              "relres_true": v["relres_true"],
                              "kind": "rocSPARSE CSR SpMV (adaptive) + rocBLAS dots, host loop"}
    log(f"{name} vendor: {v['ms_solve']:.3f} ms, {v['iterations']} it")
    A.close()
    del d_b, d_x
    if cpu:
        O = _oracle()
        host = host_cpu()
        th = host["threads"]
        capped = n >= 1000000
        cap = 50 if capped else 20000
        T = O.tiles(16, n, n, rp, ci, va)
        solve = O.bicgstab if spmvs == 2 else O.cg
        psolve = O.petsc_bcgs if spmvs == 2 else O.petsc_cg
        t0 = time.perf_counter()
        xo, rep = solve(rp, ci, va, b, TOL, cap, tiles=T, nthreads=th)
        dt = (time.perf_counter() - t0) * 1e3
        del T
        t0 = time.perf_counter()
        _, prep = psolve(rp, ci, va, b, TOL, cap, nthreads=th)
        dp = (time.perf_counter() - t0) * 1e3
        out["cpu_baseline"] = {
            "tile_solver": {"ms": round(dt, 3), "iterations": rep.iterations, "converged": bool(rep.converged),
                            "ms_per_iteration": round(dt / max(rep.iterations, 1), 4),
                            "relres_true": rep.relres_true, "kind": "port"},
            "petsc": {"ms": round(dp, 3), "iterations": prep.iterations, "converged": bool(prep.converged),
                      "ms_per_iteration": round(dp / max(prep.iterations, 1), 4),
                      "relres_true": prep.relres_true, "kind": "port (PETSc algorithm restated)"},
            "threads": th, "host": host,
            "sample": (f"capped at {cap} iterations (time per iteration reported)" if capped
                       else "full solve to true relres 1e-10"),
        }
        if not capped and rep.converged:
            out["cpu_baseline"]["gpu_err_vs_oracle_x"] = {
                k2: float(np.linalg.norm(v2 - xo) / np.linalg.norm(xo)) for k2, v2 in xsol.items()}
        log(f"{name} cpu: tile {dt:.1f} ms ({rep.iterations} it), petsc {dp:.1f} ms ({prep.iterations} it), "
            f"{th} threads")
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--grid", type=int, default=128)
    ap.add_argument("--rr", type=float, default=1e-4, help="residual replacement factor (mixed)")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-batched", action="store_true", help="skip the batched (512 systems x 8 RHS) measurement")
    ap.add_argument("--calib", action="store_true",
                    help="also run a plain 512 MiB device copy (known bytes) to calibrate PMC byte counters")
    ap.add_argument("--only-batched", action="store_true",
                    help="profiling aid: only the batched measurement; prints its record, not the bench line")
    ap.add_argument("--batched-no-tune", action="store_true", help="batched solves on the default assignment")
    ap.add_argument("--only-bicgstab", action="store_true",
                    help="profiling aid: only the 96^3 convection-diffusion BiCGSTAB record (--only-config "
                         "convdiff96_bicgstab)")
    ap.add_argument("--only-config", default=None,
                    help="profiling aid: only this workload's record (laplace256_cg, convdiff96_bicgstab, "
                         "random_spd_1m_cg); prints it, not the bench line")
    ap.add_argument("--no-configs", action="store_true",
                    help="skip the records of the other single-system workloads")
    args = ap.parse_args()
    if args.only_bicgstab:
        args.only_config = "convdiff96_bicgstab"
    if args.gpus != 1:
        print(f"bench.py: this build measures one GPU only (asked for --gpus {args.gpus}); "
              "row-block sharding over several GPUs is designed but not built", file=sys.stderr)
        sys.exit(2)

    import torch
    from __graft_entry__ import load_package

    mf = load_package()
    if not torch.cuda.is_available():
        raise RuntimeError("bench.py needs the GPU")
    rc = mf.lib().mf_init(0)
    if rc != 0:
        raise RuntimeError(mf.lib().mf_last_error().decode())

    if args.only_config:
        res = config_run(mf, torch, args.only_config, args.steps, args.warmup, cpu=not args.no_cpu)
        if args.calib:
            calibration_copy(torch)
        print(json.dumps(res), flush=True)
        return

    if args.only_batched:
        res = batched_run(mf, tune=not args.batched_no_tune)
        if args.calib:
            calibration_copy(torch)
        print(json.dumps(res), flush=True)
        return

    g = args.grid
    t0 = time.perf_counter()
    rp, ci, va = mf.gen_poisson3d(g, g, g)
    n = len(rp) - 1
    xs = mf.gen_uniform(0, n, -1.0, 1.0)
    import scipy.sparse as sp
    b = sp.csr_matrix((va, ci, rp), shape=(n, n)) @ xs
    log(f"generated n={n} nnz={len(ci)} in {time.perf_counter() - t0:.1f}s")
    t0 = time.perf_counter()
    A = mf.Matrix(rp, ci, va)
    A.layout(0.0)  # lossless per-tile classes
    info = A.info()
    log(f"tiles built on the GPU in {time.perf_counter() - t0:.1f}s: tilenum={info['tilenum']} "
        f"codes={info['tiles_per_code']}")

    dev = torch.device("cuda:0")
    npad = info["tilem"] * info["B"]
    d_b = torch.zeros(npad, dtype=torch.float64, device=dev)
    d_b[:n] = torch.from_numpy(b).to(dev)
    d_x = torch.zeros(npad, dtype=torch.float64, device=dev)
    torch.cuda.synchronize()

    def run(precision, steps, warmup):
        opts = dict(method=mf.MF_CG, tol=TOL, precision=precision)
        if precision == mf.MF_MIXED:
            opts.update(tau=0.0, rr_factor=args.rr)
        for _ in range(warmup):
            mf_rep = A.solve_device(d_b.data_ptr(), d_x.data_ptr(), **opts)
        torch.cuda.synchronize()
        reps = []
        t0 = time.perf_counter()
        for _ in range(steps):
            reps.append(A.solve_device(d_b.data_ptr(), d_x.data_ptr(), **opts))
        torch.cuda.synchronize()
        wall = (time.perf_counter() - t0) * 1e3 / steps
        for r in reps:
            if r["status"] != 0 or r["relres_true"] > TOL:
                raise RuntimeError(f"solve did not reach tolerance: {r}")
        return reps, wall

    reps64, wall64 = run(mf.MF_FP64, args.steps, args.warmup)
    x64 = d_x[:n].cpu().numpy()
    repsmx, wallmx = run(mf.MF_MIXED, args.steps, args.warmup)
    xmx = d_x[:n].cpu().numpy()
    ms64 = statistics.median(r["ms_solve"] for r in reps64)
    msmx = statistics.median(r["ms_solve"] for r in repsmx)
    it64, itmx = reps64[0]["iterations"], repsmx[0]["iterations"]
    err64 = float(np.linalg.norm(x64 - xs) / np.linalg.norm(xs))
    errmx = float(np.linalg.norm(xmx - xs) / np.linalg.norm(xs))
    log(f"fp64: {ms64:.3f} ms, {it64} it; mixed: {msmx:.3f} ms, {itmx} it, "
        f"{repsmx[0]['replacements']} true-residual passes")

    if args.calib:
        calibration_copy(torch)

    info = A.info()  # both layouts are built by now
    # standalone SpMV kernel
    spmv64 = A.spmv_bench(50, mixed=False)
    spmvmx = A.spmv_bench(50, mixed=True)
    b64, bmx = info["bytes_alg_fp64"], info["bytes_alg_mixed"]

    # phases of an iteration of the persistent solver: one more (untimed)
    # solve of each kind with workgroup 0's phase clock on.  Its SpMV ends before
    # the slowest workgroups', whose rest it books as sync, so no rate follows
    # from these times; the launch's is in the roofline
    def phase(precision):
        opts = dict(method=mf.MF_CG, tol=TOL, precision=precision, profile=1)
        if precision == mf.MF_MIXED:
            opts.update(tau=0.0, rr_factor=args.rr)
        r = A.solve_device(d_b.data_ptr(), d_x.data_ptr(), **opts)
        us = r["phase_us"]
        return {"us_per_iteration": {"spmv": round(us[0], 2), "sync_after_spmv": round(us[1], 2),
                                     "update": round(us[2], 2), "sync_after_update": round(us[3], 2)}}
    phases = {"fp64": phase(mf.MF_FP64), "mixed": phase(mf.MF_MIXED)}

    # vendor-library baseline on the same system: rocSPARSE SpMV + rocBLAS
    # dots in a host loop (as the reference's hipSPARSE driver), FP64 CG to
    # the same true relative residual
    vreps = [A.vendor_solve_device(d_b.data_ptr(), d_x.data_ptr(), method=mf.MF_CG, tol=TOL) for _ in range(3)]
    for r in vreps:
        if r["status"] != 0 or r["relres_true"] > TOL:
            raise RuntimeError(f"vendor baseline did not reach tolerance: {r}")
    vms = statistics.median(r["ms_solve"] for r in vreps)
    vendor = {"ms": round(vms, 4), "iterations": vreps[0]["iterations"], "relres_true": vreps[0]["relres_true"],
              "kind": "rocSPARSE CSR SpMV (adaptive) + rocBLAS ddot, host loop with a residual read per iteration",
              "speedup_mixed": round(vms / msmx, 3), "speedup_fp64": round(vms / ms64, 3)}
    log(f"vendor CG: {vms:.3f} ms, {vreps[0]['iterations']} it (mixed {vendor['speedup_mixed']}x, "
        f"fp64 {vendor['speedup_fp64']}x faster)")
    log(f"phases of an iteration, us, workgroup 0's clock: {phases}")

    # dominant kernel: the persistent CG launch (one per solve).  Unit = one
    # SpMV at its algorithmic bytes B_alg (values and indices at their stored
    # widths, tile metadata, the gathered vector read once, y written once);
    # the solve runs one SpMV per iteration.  The other Krylov vectors stay in
    # registers and LDS for the whole solve and are not counted, nor are the
    # true-residual passes.
    traffic = None
    pmc_file = os.path.join(ROOT, "profiles", "k_cg_poisson128_pmc.json")
    if g == 128 and os.path.exists(pmc_file):
        with open(pmc_file) as f:
            pmc = json.load(f)
        # calibrated FETCH_SIZE + WRITE_SIZE of the mixed launch, per iteration
        traffic = round(pmc["mixed"]["traffic_bytes_per_iteration"] * itmx)
    iw = info["index_width"]
    # the 7-point system runs on stencil planes: values without indices
    roof = _roofline(itmx, 1, bmx, msmx)
    roof.update({
        "traffic": traffic,
        "kernel": f"k_cg<Stencil<3,7>,512,{repsmx[0]['rows_per_thread']}> (persistent mixed CG on E4M3 stencil planes, "
                  "one launch per solve)",
        "unit_def": "one SpMV at B_alg (SpMV algorithmic bytes of the mixed layout); one per CG iteration",
        "launch_ms": round(msmx, 4),
        "per_step_GBps": round(itmx * bmx / (wallmx * 1e-3) / 1e9, 1),
        "fp64": _roofline(it64, 1, b64, ms64),
        "traffic_source": "profiles/k_cg_poisson128_pmc.json (rocprofv3 FETCH_SIZE, WRITE_SIZE, calibrated "
                          "against a device copy of known size)" if traffic is not None else None,
    })
    if roof["achieved"] > HBM_PEAK / 1e9 or roof["per_step_GBps"] > HBM_PEAK / 1e9:
        raise RuntimeError(f"algorithmic rate above the HBM peak: {roof}")

    A.close()
    del d_b, d_x
    batched = None if args.no_batched else batched_run(mf)

    configs = None
    if not args.no_configs:
        configs = {name: config_run(mf, torch, name, args.steps, args.warmup, cpu=not args.no_cpu)
                   for name in _configs(mf)}

    cpu = None
    if not args.no_cpu:
        log("cpu baseline ...")
        cpu = cpu_baseline(rp, ci, va, b, it64, {"fp64": x64, "mixed": xmx})
        log(f"cpu: {cpu['value']} ms (oracle tile CG), {cpu['petsc_cg']['ms']} ms (PETSc CG restatement); "
            f"GPU x vs oracle x: {cpu['gpu_err_vs_oracle_x']}")

    out = {
        "metric": METRIC,
        "value": round(msmx, 4),
        "unit": "ms",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(wallmx, 4),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64 vectors/dots; e4m3 tiles, f32 accumulation",
        "data": "synthetic",
        "config": {
            "workload": f"3D 7-point Poisson {g}^3, CG to true relres 1e-10, b = A x*, x* ~ U(-1,1) seed 0",
            "n": n, "nnz": int(len(ci)), "tile": 16, "precision": "per-tile mixed (lossless: all tiles E4M3)",
            "iterations_mixed": itmx, "iterations_fp64": it64,
            "replacements_mixed": repsmx[0]["replacements"],
            "grid": repsmx[0]["grid"], "block": repsmx[0]["block"],
            "rows_per_thread": repsmx[0]["rows_per_thread"],
            "index_width": iw,
            "pattern_slabs": {"fp64": info["pattern_slabs_fp64"], "mixed": info["pattern_slabs_mixed"],
                              "tile_rows": info["tilem"]},
        },
        "fp64_ms": round(ms64, 4),
        "fp64_ms_per_step_wall": round(wall64, 4),
        "speedup_mixed_vs_fp64": round(ms64 / msmx, 3),
        "relres_true": {"fp64": reps64[0]["relres_true"], "mixed": repsmx[0]["relres_true"]},
        "err_vs_xstar": {"fp64": err64, "mixed": errmx},
        "spmv": {
            "fp64": {"ms": round(spmv64, 5), "GB/s": round(b64 / spmv64 / 1e6, 1),
                     "frac": round(b64 / (spmv64 * 1e-3) / HBM_PEAK, 4), "bytes_alg": b64},
            "mixed": {"ms": round(spmvmx, 5), "GB/s": round(bmx / spmvmx / 1e6, 1),
                      "frac": round(bmx / (spmvmx * 1e-3) / HBM_PEAK, 4), "bytes_alg": bmx},
        },
        "spmv_phase_in_solver": phases,
        "vendor_baseline": vendor,
        "roofline": roof,
        "batched": batched,
        "cpu_baseline": cpu,
        "configs": configs,
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
