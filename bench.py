#!/usr/bin/env python3
"""Benchmark of the MI355X deviational MC engine.

Workload (one "step" of this benchmark = one full beRTAMC2D transient run
of R independent replicas, R = 4 by default): 2000-mode synthetic material,
synthetic energy-conserving collision operator (5% dense), propagator
P = exp(5 ps * B) built on the GPU by the block-Krylov path (FP64, m = 30);
per replica a 500 nm x 100 nm ribbon in 50 x-bins, 1 K pulse in bin 0 giving
~1e6 deviational particles, 200 time steps of 5 ps with adiabatic diffuse
walls and cancellation every 4 steps. The R replicas are disjoint copies of
the ribbon in one geometry (they share no side), so one run advances R
independent replicas together; sigma(T) comes from all replicas of all timed
runs (seed = base + step).

value = particle-events/s over the timed steps, where a particle-event of
beRTAMC2D is one particle advected and scattered for one time step.

Extras (not the headline value): RTAMC2D at the 3000-mode, 1e6-particle
steady-state configuration (events/s) and the Krylov propagator build at
N = 8192, m = 30 in FP32 / BF16 against FP64.
"""
import argparse
import ctypes
import json
import os
import platform
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
BYTES_PER_PARTICLE_STEP = 72  # 32 B state in + 32 B out + 8 B propagator alias entry


def load_pkg():
    import importlib.util
    name = "bte_barna_amd"
    if name in sys.modules:
        return sys.modules[name]
    path = os.path.join(ROOT, "bte-barna_amd", "__init__.py")
    spec = importlib.util.spec_from_file_location(name, path, submodule_search_locations=[os.path.dirname(path)])
    mod = importlib.util.module_from_spec(spec)
    sys.modules[name] = mod
    spec.loader.exec_module(mod)
    return mod


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def measured_traffic():
    """HBM bytes per step-kernel launch from the committed rocprofv3 PMC
    summary (FETCH_SIZE + WRITE_SIZE scaled by the copy-kernel factor)."""
    path = os.path.join(ROOT, "profiles", "bert_step_kernel_pmc.json")
    if not os.path.exists(path):
        return None
    with open(path) as f:
        d = json.load(f)
    return d.get("hbm_bytes_per_launch")


def host_cpus():
    """Threads the CPU baselines use and what the host has: the process's
    CPU allotment (OMP_NUM_THREADS where the launcher sets it, else the CPUs
    this process may run on), os.cpu_count() and the CPU model name as
    /proc/cpuinfo (lscpu's source) gives it."""
    try:
        affinity = len(os.sched_getaffinity(0))
    except AttributeError:
        affinity = os.cpu_count()
    env = int(os.environ.get("OMP_NUM_THREADS", "0") or 0)
    model = platform.processor() or platform.machine()
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    threads = env if env > 0 else affinity
    return {"threads": threads, "nproc": os.cpu_count(), "affinity": affinity, "omp_num_threads": env or None,
            "model": model}


def _oracle():
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_lib as orc
    return orc


def _with_host(d, host, one):
    """adds the host description and the 1-thread figure to a baseline"""
    d.update({"cores": host["threads"], "nproc": host["nproc"], "affinity": host["affinity"],
              "cpu_model": host["model"], "value_1thread": one["value"], "sample_1thread": one["sample"]})
    return d


def cpu_baseline(pkg, mat, P, cfg, nparticles, nsteps):
    """The oracle (C++ restatement of the reference loop, OpenMP) on a bounded
    sample of the same workload: fewer initial particles and steps; on every
    allotted thread, and on one thread over a tenth of the particles and a
    quarter of the steps."""
    orc = _oracle()
    host = host_cpus()

    def leg(npart, nst, nthreads):
        t0 = time.perf_counter()
        o = orc.bert_run(mat, cfg["rect"], cfg["kind"], cfg["Teq"], cfg["Tinit"], thickness=cfg["thickness"],
                         dt=cfg["dt"], maxtime=cfg["dt"] * (nst - 1), P=P, Efactor=npart,
                         Tmax=cfg["Tmax"], Tmin=cfg["Tmin"], seed=12345, max_steps=nst, nthreads=nthreads)
        el = time.perf_counter() - t0
        ps = int(o["npart"][:-1].sum())  # particles entering each step
        return {"value": ps / el, "sample": f"oracle beRTAMC2D, same material/propagator/geometry, {npart} initial "
                                            f"particles x {nst} steps ({ps} particle-events in {el:.2f} s)"}

    full = leg(nparticles, nsteps, host["threads"])
    one = leg(max(1, nparticles // 10), max(2, nsteps // 4), 1)
    return _with_host({"value": full["value"], "unit": "particle-events/s", "kind": "port",
                       "sample": full["sample"]}, host, one)


def rta_cpu_baseline(c, nparticles):
    """The oracle's RTAMC2D history loop (OpenMP over particles) on a bounded
    particle sample of configuration 0; on every allotted thread, and on one
    thread over a tenth of the particles."""
    orc = _oracle()
    host = host_cpus()

    def leg(npart, nthreads):
        t0 = time.perf_counter()
        o = orc.rta_run(c["material"], c["rect"], c["kind"], c["Teq"], thickness=c["thickness"], T0=c["T0"],
                        dt=c["dt"], maxtime=c["maxtime"], nparticles=npart, seed=12345, sigma=c["sigma_bounce"],
                        nthreads=nthreads)
        el = time.perf_counter() - t0
        return {"value": o["events"] / el, "sample": f"oracle RTAMC2D, configuration 0 with {npart} particles "
                                                     f"({o['events']} events in {el:.2f} s)"}

    full = leg(nparticles, host["threads"])
    one = leg(max(1, nparticles // 10), 1)
    return _with_host({"value": full["value"], "unit": "particle-events/s", "kind": "port",
                       "sample": full["sample"]}, host, one)


def single_replica(pkg, ctx, modes, prop, cfg1, steps):
    """Configuration 1 as stated: one ribbon, ~1e6 initial particles, one run
    per timed step (the headline advances several replicas per run)."""
    geom = pkg.Geometry(ctx, cfg1["rect"], cfg1["kind"], cfg1["Teq"], cfg1["Tinit"])
    runs = [pkg.BertRun(ctx, modes, geom, prop, thickness=cfg1["thickness"], dt=cfg1["dt"], maxtime=cfg1["maxtime"],
                        max_steps=cfg1["max_steps"], Efactor=cfg1["Efactor"], Tmax=cfg1["Tmax"], Tmin=cfg1["Tmin"],
                        seed=5000 + s) for s in range(steps + 1)]
    runs[0].execute()
    ctx.sync()
    t0 = time.perf_counter()
    ev = sum(r.execute()["particle_steps"] for r in runs[1:])
    ctx.sync()
    el = time.perf_counter() - t0
    for r in runs:
        r.close()
    geom.close()
    return {"workload": "configuration 1, one replica per run", "runs": steps, "seconds": el,
            "ms_per_run": el / steps * 1e3, "particle_events_per_s": ev / el}


def rta_extra(pkg, ctx, cpu_particles=0):
    W = pkg.workloads
    c = W.config0()
    m = c["material"]
    modes = pkg.ModeTable(ctx, m["omega"], m["vx"], m["vy"], m["w"], m["V"], m["lattz"])
    geom = pkg.Geometry(ctx, c["rect"], c["kind"], c["Teq"])
    r = pkg.RtaRun(ctx, modes, geom, thickness=c["thickness"], T0=c["T0"], dt=c["dt"], maxtime=c["maxtime"],
                   nparticles=c["nparticles"], seed=1, sigma_bounce=c["sigma_bounce"])
    r.execute()  # warm-up
    ctx.sync()
    t0 = time.perf_counter()
    out = r.execute()
    el = time.perf_counter() - t0
    r.close()
    T = out["T"][-1, :100]
    # sigma(T) at the final time over R = 16 independent replicas (disjoint
    # seeds), run as one batch: the particle count that meets a 2 mK target
    R = 16
    b = pkg.RtaBatch(ctx, modes, [dict(geom=geom, T0=c["T0"], nparticles=c["nparticles"], seed=100 + k)
                                  for k in range(R)],
                     thickness=c["thickness"], dt=c["dt"], maxtime=c["maxtime"], sigma_bounce=c["sigma_bounce"],
                     tally="fp64-lds-runs")
    b.execute()
    ctx.sync()
    t0 = time.perf_counter()
    res, rep = b.execute()
    t_rep = time.perf_counter() - t0
    b.close()
    Tl = np.array([o["T"][-1, :100] for o in res])
    sig = float((Tl.std(0, ddof=1) / np.sqrt(R)).max())
    return {"workload": "RTAMC2D steady state: 3000 modes, 1e6 particles, 1 um x 200 nm, +-0.5 K walls, 100 x-bins, "
                        "dt 25 ps, maxtime 5 ns",
            "events": int(out["events"]), "crossings": int(out["crossings"]), "seconds": el,
            "events_per_s": out["events"] / el, "kernel_ms": out["kernel_ms"],
            "kernel_events_per_s": out["events"] / (out["kernel_ms"] * 1e-3),
            "T_left_right": [float(T[0]), float(T[-1])],
            "sigma_T": {"replicas": R, "particles_per_replica": c["nparticles"], "max_bin_sigma_K": sig,
                        "target_K": 0.002, "met": sig <= 0.002, "seconds": t_rep,
                        "events_per_s": rep["events"] / t_rep, "tally": "fp64-lds-runs (mode 3)"},
            **({"cpu_baseline": rta_cpu_baseline(c, cpu_particles)} if cpu_particles else {})}


def batch_extra(pkg, ctx):
    """64 independent RTAMC2D runs (widths 50 nm - 2 um, 100 - 500 K, 1e5 - 1e7
    particles) in one graph-replayed launch with FP64 LDS tallies per run
    (tally mode 3), against the same batch with FP64 device-atomic tallies
    (mode 0, tuned launch shape) and against the 64 runs launched one after
    another, each with its best single-run tallies (mode 2)."""
    W = pkg.workloads
    c = W.config3()
    m = c["material"]
    modes = pkg.ModeTable(ctx, m["omega"], m["vx"], m["vy"], m["w"], m["V"], m["lattz"])
    runs = []
    for r in c["runs"]:
        runs.append(dict(geom=pkg.Geometry(ctx, r["rect"], r["kind"], r["Teq"]), T0=r["T0"],
                         nparticles=r["nparticles"], seed=r["seed"], wscale=r["wscale"]))
    kw = dict(thickness=c["thickness"], dt=c["dt"], maxtime=c["maxtime"], sigma_bounce=c["sigma_bounce"])
    b = pkg.RtaBatch(ctx, modes, runs, use_graph=True, tally="fp64-lds-runs", **kw)
    b.execute()  # captures the graph
    ctx.sync()
    t0 = time.perf_counter()
    res, rep = b.execute()
    t_batch = time.perf_counter() - t0
    b.close()
    # the same batch with device-atomic tallies and a tuned launch shape
    a = pkg.RtaBatch(ctx, modes, runs, use_graph=True, **kw)
    block, blocks = a.tune(fraction=0.02)
    ctx.sync()
    t0 = time.perf_counter()
    res0, rep0 = a.execute()
    t_atomics = time.perf_counter() - t0
    a.close()
    same = (int(rep0["events"]), int(rep0["crossings"])) == (int(rep["events"]), int(rep["crossings"]))
    dT = max(float(np.abs(x["T"] - y["T"]).max()) for x, y in zip(res, res0))
    # plain form: each run in its own launch
    t_seq, ev_seq = 0.0, 0
    for r in runs:
        s = pkg.RtaBatch(ctx, modes, [r], tally="fp64-lds", **kw)
        t0 = time.perf_counter()
        _, rr = s.execute()
        t_seq += time.perf_counter() - t0
        ev_seq += rr["events"]
        s.close()
    L = c["length"] * 1e-9
    kappa = [float(o["jx"][-1, :100].mean() * L / 1.0) for o in res]
    return {"workload": "64 RTAMC2D runs: widths 50 nm-2 um (log), 100-500 K, 1e5-1e7 particles (seeded), "
                        "3000 modes, 1 um long, 100 bins, dt 25 ps, maxtime 5 ns, tau ~ 1/T",
            "particles": int(sum(r["nparticles"] for r in runs)), "events": int(rep["events"]),
            "batched_s": t_batch, "batched_kernel_ms": rep["kernel_ms"], "tally": "fp64-lds-runs (mode 3)",
            "batched_events_per_s": rep["events"] / t_batch,
            "batched_fp64_atomics_s": t_atomics, "fp64_atomics_launch": [block, blocks],
            "same_histories_as_fp64_atomics": bool(same), "max_abs_T_diff_vs_fp64_atomics_K": dT,
            "sequential_s": t_seq, "sequential_tally": "fp64-lds (mode 2) per run",
            "speedup_vs_sequential": t_seq / t_batch,
            "kappa_W_per_mK": {"first": kappa[0], "last": kappa[-1], "min": min(kappa), "max": max(kappa)}}


def grad_extra(pkg, ctx, fd_dp=0.01, seeds=8):
    """Differentiable transient RTAMC2D: T(x, t) and dT/dp_top, dT/dp_bottom
    from one run with score-function tallies, against plain runs and a
    central-difference estimate with common random numbers. Plain and
    gradient runs are timed with both tally modes: FP64 device atomics, and
    FP32 per-workgroup partial sums in LDS with an FP64 final sum. Over
    `seeds` independent seeds (each: one gradient run and four
    central-difference runs on the same streams) the two estimators of the
    left-half mean temperature derivative get means and standard errors on
    both edges."""
    W = pkg.workloads
    c = W.config4()
    m = c["material"]
    modes = pkg.ModeTable(ctx, m["omega"], m["vx"], m["vy"], m["w"], m["V"], m["lattz"])
    geom = pkg.Geometry(ctx, c["rect"], c["kind"], c["Teq"])
    kw = dict(thickness=c["thickness"], dt=c["dt"], maxtime=c["maxtime"], sigma_bounce=c["sigma_bounce"])
    base = dict(geom=geom, T0=c["T0"], nparticles=c["nparticles"], seed=c["seed"])
    p = np.array(c["specularity"])
    times, outs, events = {}, {}, 0
    for tally in ("fp64", "fp32-lds"):
        for grad in (False, True):
            b = pkg.RtaBatch(ctx, modes, [dict(base, specularity=tuple(p), grad=grad)], tally=tally, **kw)
            b.execute(grad=grad)  # warm-up
            t0 = time.perf_counter()
            (o,), rep = b.execute(grad=grad)
            times[(tally, grad)] = time.perf_counter() - t0
            outs[(tally, grad)] = o
            events = int(rep["events"])
            b.close()
    obs = lambda T: float(T[-1, :64].mean())  # left half, last time
    sides = ((2, "top"), (1, "bottom"))
    score = {n: [] for _, n in sides}
    fdiff = {n: [] for _, n in sides}
    for k in range(seeds):
        sd = dict(base, seed=1000 + k)
        g = pkg.RtaBatch(ctx, modes, [dict(sd, specularity=tuple(p), grad=True)], tally="fp32-lds", **kw)
        (go,), _ = g.execute(grad=True)
        g.close()
        for side, name in sides:
            score[name].append(obs(go["dTdp"][side]))
            T = []
            for sgn in (+1, -1):
                q = p.copy()
                q[side] += sgn * fd_dp
                f = pkg.RtaBatch(ctx, modes, [dict(sd, specularity=tuple(q))], tally="fp32-lds", **kw)
                (fo,), _ = f.execute()
                f.close()
                T.append(obs(fo["T"]))
            fdiff[name].append((T[0] - T[1]) / (2 * fd_dp))
    t_plain = times[("fp32-lds", False)]
    t_grad = times[("fp32-lds", True)]
    out, ratio = {}, 0.0
    for _, name in sides:
        a, b_ = np.array(score[name]), np.array(fdiff[name])
        se_a, se_b = a.std(ddof=1) / np.sqrt(seeds), b_.std(ddof=1) / np.sqrt(seeds)
        d = a - b_
        out[name] = {"score_mean_K": float(a.mean()), "score_se_K": float(se_a),
                     "central_fd_mean_K": float(b_.mean()), "central_fd_se_K": float(se_b),
                     "paired_difference_K": float(d.mean()), "paired_difference_se_K": float(d.std(ddof=1) / np.sqrt(seeds)),
                     "z": float(d.mean() / (d.std(ddof=1) / np.sqrt(seeds)))}
        ratio = max(ratio, (se_b / se_a) ** 2)
    g64 = outs[("fp64", True)]
    go = outs[("fp32-lds", True)]
    return {"workload": "1 um x 100 nm, 128 bins x 64 time bins, 5000 mirror-pair modes, 1e7 particles, "
                        "p_top 0.3, p_bottom 0.7, walls 300 +- 0.5 K",
            "runs_s": {f"{t}_{'grad' if g else 'plain'}": v for (t, g), v in times.items()},
            "grad_run_s": t_grad, "plain_run_s": t_plain, "events": events,
            "useful_run_speedup": 5 * t_plain / t_grad,
            "useful_run_speedup_equal_se": (t_plain + 4 * t_plain * ratio) / t_grad,
            "fd_over_score_variance": ratio,
            "fp32_vs_fp64_tallies": {
                "max_abs_T_diff_K": float(np.abs(go["T"] - g64["T"]).max()),
                "max_abs_dTdp_diff_K": float(np.abs(go["dTdp"] - g64["dTdp"]).max())},
            "note": "both forms with FP32 LDS tallies; per run, one gradient run replaces the base run and four "
                    "central-difference runs (at most 5x); at equal standard error of dT/dp the four "
                    "central-difference runs are repeated (se_fd / se_score)^2 times",
            "derivatives": out, "seeds": seeds, "fd_dp": fd_dp}


def krylov_extra(pkg, ctx, N=8192, m=30, cpu_cols=0):
    W = pkg.workloads
    mat, B = W.config1_inputs(nmodes=N, seed=1)
    res = {}
    # the first build of each precision loads the BLAS kernels for that shape;
    # it is timed separately and the second build is reported
    first = {}
    for prec in ("fp64", "fp32", "bf16"):
        _, r0 = pkg.build_P(ctx, B, 5.0, m=2, precision=prec, arnoldi="textbook")
        first[prec] = r0["build_ms"]
    # FP64 Pade exponential on the GPU as the exact reference
    Ex, ex_ms = pkg.expm(ctx, B, 5.0)
    res["pade_expm_fp64_ms"] = ex_ms
    P64, rep64 = pkg.build_P(ctx, B, 5.0, m=m, precision="fp64", arnoldi="textbook")
    res["fp64"] = {"build_ms": rep64["build_ms"], "gemm_ms": rep64["gemm_ms"], "gemm_tflops": rep64["gemm_tflops"],
                   "col_sum_drift": rep64["max_col_sum_err"],
                   "max_col_L1_vs_pade": float(np.abs(P64 - Ex).sum(0).max())}
    Pr, repr_ = pkg.build_P(ctx, B, 5.0, m=m, precision="fp64", arnoldi="reference")
    res["fp64_reference_arnoldi"] = {"build_ms": repr_["build_ms"],
                                     "max_col_L1_vs_pade": float(np.abs(Pr - Ex).sum(0).max()),
                                     "max_col_L1_vs_fp64": float(np.abs(Pr - P64).sum(0).max()),
                                     "col_sum_drift": float(np.abs(Pr.sum(0) - 1).max())}
    del Pr
    res["first_call_ms_m2"] = first
    for prec in ("fp32", "bf16"):
        P, rep = pkg.build_P(ctx, B, 5.0, m=m, precision=prec, arnoldi="textbook")
        res[prec] = {"build_ms": rep["build_ms"], "gemm_ms": rep["gemm_ms"], "gemm_tflops": rep["gemm_tflops"],
                     "max_col_L1_vs_fp64": float(np.abs(P - P64).sum(0).max()),
                     "max_col_L1_vs_pade": float(np.abs(P - Ex).sum(0).max()),
                     "col_sum_drift_before_projection": rep["max_col_sum_err"],
                     "col_sum_drift_after": float(np.abs(P.sum(0) - 1).max())}
        del P
    del Ex
    res["workload"] = f"PropagatorBuilder Krylov N={N}, m={m}, dt=5 ps, all columns as block-Krylov GEMMs"
    res["flops_2mN3"] = 2.0 * m * N ** 3
    if cpu_cols:
        log(f"extra: Krylov CPU sample ({cpu_cols} columns) ...")
        res["cpu_baseline"] = krylov_cpu_baseline(B, m, cpu_cols, res["fp64_reference_arnoldi"]["build_ms"])
    return res


def krylov_cpu_baseline(B, m, ncols, gpu_ms):
    """The oracle's per-column FP64 Arnoldi + Pade (OpenMP over columns, the
    reference's build_P loop) on a bounded sample of columns, extrapolated to
    all N columns; compared with the GPU build of the same Arnoldi."""
    orc = _oracle()
    host = host_cpus()
    N = B.shape[0]
    A = np.asfortranarray(B)

    def leg(nc, nthreads):
        t0 = time.perf_counter()
        orc.build_P_cols(A, 5.0, m, 0, 0, nc, nthreads)
        el = time.perf_counter() - t0
        return {"value": el * N / nc,
                "sample": f"oracle build_P, reference Arnoldi, FP64, columns 0..{nc - 1} of {N} in {el:.2f} s"}

    full = leg(ncols, host["threads"])
    one = leg(max(1, ncols // 8), 1)
    d = _with_host({"value": full["value"], "unit": "s per full propagator (extrapolated)", "kind": "port",
                    "sample": full["sample"]}, host, one)
    d.update({"gpu_fp64_reference_arnoldi_s": gpu_ms * 1e-3, "gpu_speedup": full["value"] / (gpu_ms * 1e-3),
              "gpu_speedup_vs_1thread": one["value"] / (gpu_ms * 1e-3)})
    return d


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-extras", action="store_true")
    ap.add_argument("--cpu-particles", type=int, default=1_000_000)
    ap.add_argument("--cpu-steps", type=int, default=200)
    ap.add_argument("--replicas", type=int, default=4, help="independent replicas advanced together per run")
    ap.add_argument("--extra", choices=("rta_steady", "rta_batch", "rta_grad", "krylov"),
                    help="run only this extra measurement and print its JSON (for profiling one workload)")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run a plain 1 GiB device copy (scale reference for rocprofv3 FETCH_SIZE/WRITE_SIZE)")
    args = ap.parse_args()
    if args.copy_calibration:
        import torch
        x = torch.ones(256 * 1024 * 1024, dtype=torch.float32, device="cuda")
        y = torch.empty_like(x)
        for _ in range(3):
            y.copy_(x)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes": x.numel() * 4, "copies": 3}), flush=True)
        return
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (asked for {args.gpus}); the engine runs on a single GPU and "
              f"multi-GPU sharding is not part of this build.", file=sys.stderr)
        sys.exit(2)

    pkg = load_pkg()
    W = pkg.workloads
    ctx = pkg.Context(0)
    if args.extra:
        fn = {"rta_steady": rta_extra, "rta_batch": batch_extra, "rta_grad": grad_extra,
              "krylov": krylov_extra}[args.extra]
        print(json.dumps({"extra": args.extra, **fn(pkg, ctx)}), flush=True)
        return
    log("setup: material, collision operator, propagator")
    mat, B = W.config1_inputs()
    P, krep = pkg.build_P(ctx, B, 5.0, m=30, precision="fp64", arnoldi="textbook")
    cfg = W.config1(replicas=args.replicas)
    cfg1 = W.config1()
    modes = pkg.ModeTable(ctx, mat["omega"], mat["vx"], mat["vy"], mat["w"], mat["V"], mat["lattz"])
    geom = pkg.Geometry(ctx, cfg["rect"], cfg["kind"], cfg["Teq"], cfg["Tinit"])
    prop = pkg.Propagator(ctx, P)
    runs = []
    for s in range(args.warmup + args.steps):
        runs.append(pkg.BertRun(ctx, modes, geom, prop, thickness=cfg["thickness"], dt=cfg["dt"],
                                maxtime=cfg["maxtime"], max_steps=cfg["max_steps"], Efactor=cfg["Efactor"],
                                Tmax=cfg["Tmax"], Tmin=cfg["Tmin"], seed=1000 + s))
    for s in range(args.warmup):
        runs[s].execute()
        log(f"warmup {s} done")
    ctx.sync()
    t0 = time.perf_counter()
    outs = []
    for s in range(args.warmup, args.warmup + args.steps):
        outs.append(runs[s].execute())
    ctx.sync()
    elapsed = time.perf_counter() - t0
    log(f"timed {args.steps} runs in {elapsed:.3f} s")
    events = sum(o["particle_steps"] for o in outs)
    value = events / elapsed
    # HIP events bracket one step-kernel launch in 16 (one in every fourth
    # cancellation cycle, each step type in turn, of equal weight in the
    # mean); the bytes are averaged over all
    k_ms = sum(o["step_kernel_ms"] for o in outs)
    k_timed = sum(o["step_kernel_timed"] for o in outs)
    k_launch = sum(o["step_kernel_launches"] for o in outs)
    k_units = sum(o["step_kernel_particle_steps"] for o in outs)
    avg_ms = k_ms / k_timed
    bytes_per_launch = BYTES_PER_PARTICLE_STEP * k_units / k_launch
    achieved = bytes_per_launch / (avg_ms * 1e-3) / 1e9
    # sigma(T) at the last step across the replicas (T = T0 + ed / Cv)
    cv = 1.6e6
    nb = len(cfg1["rect"])
    Tlast = np.array([300.0 + o["props"][-1, r * nb:(r + 1) * nb, 0] / cv for o in outs
                      for r in range(args.replicas)])
    sigmaT = float((Tlast.std(0, ddof=1) / np.sqrt(len(Tlast))).max()) if len(Tlast) > 1 else None
    conserved = all(bool(((o["npart"] + o["pending"]) == o["npart"][0]).all()) for o in outs)
    line = {
        "metric": "deviational-MC particle-events/s at fixed σ(T); Krylov propagator build time",
        "value": value,
        "unit": "particle-events/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": elapsed / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": "beRTAMC2D transient: 2000-mode synthetic material, 5%-dense synthetic Omega, "
                               "P=exp(-Omega*5ps) (GPU Krylov FP64 m=30), 500x100 nm ribbon, 50 x-bins, 1 K pulse "
                               "in bin 0, ~1e6 particles, 200 steps of 5 ps; one bench step = one full run of "
                               f"{args.replicas} independent replicas advanced together",
                   "replicas_per_run": args.replicas,
                   "initial_particles": int(outs[0]["npart"][0]), "time_steps": int(outs[0]["nsteps"]),
                   "particle_events_per_run": int(outs[0]["particle_steps"]),
                   "max_sigma_T_K_last_step": sigmaT, "count_conserved": conserved,
                   "parallelism": "single GPU"},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": measured_traffic(),
                     "kernel": "bert_step_kernel", "avg_launch_ms": avg_ms,
                     "launches_timed": k_timed, "launches": k_launch,
                     "algorithmic_bytes_per_launch": bytes_per_launch},
    }
    if not args.no_cpu:
        log("cpu baseline (oracle) ...")
        cb = cpu_baseline(pkg, mat, P, cfg1, args.cpu_particles, args.cpu_steps)
        cb["gpu_over_cpu"] = value / cb["value"]
        cb["gpu_over_cpu_1thread"] = value / cb["value_1thread"]
        line["cpu_baseline"] = cb
        log("cpu baseline done")
    if not args.no_extras:
        ex = {"config1_single_replica": single_replica(pkg, ctx, modes, prop, cfg1, args.steps)}
        log("extra: RTAMC2D config ...")
        ex["rta_steady"] = rta_extra(pkg, ctx, cpu_particles=0 if args.no_cpu else 200000)
        rs = ex["rta_steady"]
        if "cpu_baseline" in rs:
            rs["cpu_baseline"]["gpu_over_cpu"] = rs["kernel_events_per_s"] / rs["cpu_baseline"]["value"]
            rs["cpu_baseline"]["gpu_over_cpu_1thread"] = rs["kernel_events_per_s"] / rs["cpu_baseline"]["value_1thread"]
        log("extra: batched RTAMC2D sweep ...")
        ex["rta_batch"] = batch_extra(pkg, ctx)
        log("extra: specularity gradient ...")
        ex["rta_grad"] = grad_extra(pkg, ctx)
        log("extra: Krylov N=8192 ...")
        ex["krylov"] = krylov_extra(pkg, ctx, cpu_cols=0 if args.no_cpu else 32)
        ex["propagator_setup_ms"] = krep["build_ms"]
        line["extras"] = ex
    for r in runs:
        r.close()
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
