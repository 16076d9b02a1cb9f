"""Performance cases of the engine: what users of its public entry points
(RtaRun, RtaBatch, SpecularityModel, BertRun, build_P) run, from a short
trial run to the benchmark configurations, over the sizes, geometries, tally
modes, scattering models and precisions the engine takes.

A case is a dict of plain values: "kind" picks the entry point, the rest are
its sizes. prepare() makes what a user's program holds before the timed call
(mode tables, geometry, the run handle, a propagator), run() is one pass
through the entry point, exact() is the 64-bit reference where the output has
one. Monte Carlo runs have none: their outputs are a function of the seed.
The random material, the Monte Carlo seed and the operators all come from the
seed given to prepare()."""
import importlib
import math

import numpy as np
import torch

bte = importlib.import_module("bte-barna_amd")
_autograd = importlib.import_module("bte-barna_amd.autograd")

_CTX = None


def _ctx():
    """One context per process, as a user's program keeps it."""
    global _CTX
    if _CTX is None:
        _CTX = bte.Context(0)
    return _CTX


def listed():
    return [
        # a trial run of a short ribbon before a production run: the smallest
        # call, launches and the longest history
        {"name": "rta_trial", "kind": "rta", "modes": 500, "particles": 2000, "length": 200.0, "width": 50.0,
         "bins": 20, "maxtime": 500.0, "steps": 50},
        # the RTAMC2D benchmark: 1 um x 200 nm between 300 +- 0.5 K, 100 bins,
        # 200 time bins, 1e6 particles
        {"name": "rta_ribbon", "kind": "rta", "modes": 3000, "particles": 1000000, "length": 1000.0,
         "width": 200.0, "bins": 100, "maxtime": 5000.0, "steps": 200},
        # a nanoribbon with zigzag edges and slanted cells (convex polygons),
        # odd numbers of cells and modes
        {"name": "rta_zigzag", "kind": "rta_poly", "modes": 1501, "particles": 200000, "length": 370.0,
         "width": 80.0, "bins": 37, "maxtime": 1500.0, "steps": 75},
        # <spectral> output at three boxes of a ribbon
        {"name": "rta_spectral", "kind": "rta_spectral", "modes": 1000, "particles": 200000, "length": 500.0,
         "width": 100.0, "bins": 50, "maxtime": 1500.0, "steps": 60, "locations": 3, "ticks": 100},
        # a width and temperature sweep as one batch: 16 runs of uneven
        # particle counts, each run's tallies in LDS
        {"name": "rta_sweep", "kind": "rta_batch", "modes": 3000, "runs": 16, "min_particles": 30000,
         "max_particles": 1000000, "length": 1000.0, "bins": 100, "maxtime": 5000.0, "steps": 200},
        # the differentiable benchmark at a tenth of its particles: specular
        # edges with dT/dp, FP32 tallies in LDS
        {"name": "rta_edges_grad", "kind": "rta_grad", "modes": 5000, "particles": 1000000, "length": 1000.0,
         "width": 100.0, "bins": 128, "maxtime": 5000.0, "steps": 64, "p_top": 0.3, "p_bottom": 0.7},
        # one iteration of fitting the edge specularities through autograd:
        # forward and backward of T(p)
        {"name": "specularity_fit", "kind": "fit", "modes": 1000, "particles": 100000, "length": 300.0,
         "width": 60.0, "bins": 30, "maxtime": 1500.0, "steps": 30, "p_top": 0.4, "p_bottom": 0.6},
        # the beRTAMC2D benchmark's literal configuration, half its steps: one
        # ribbon with a 1 K pulse, 1e6 particles
        {"name": "bert_pulse", "kind": "bert", "modes": 2000, "particles": 1000000, "bins": 50, "replicas": 1,
         "steps": 100},
        # the beRTAMC2D benchmark's headline run: four replicas together
        {"name": "bert_replicas", "kind": "bert", "modes": 2000, "particles": 1000000, "bins": 50, "replicas": 4,
         "steps": 200},
        # a bar heated from one reservoir, periodic in y, relaxation-time
        # scattering (no propagator), odd numbers of modes and bins
        {"name": "bert_heated_rta", "kind": "bert_heated", "modes": 777, "particles": 300000, "bins": 41,
         "steps": 80},
        # PropagatorBuilder in FP64 at the size beRTAMC2D's benchmark consumes
        {"name": "krylov_fp64", "kind": "krylov", "n": 2000, "m": 30, "precision": "fp64"},
        # PropagatorBuilder's compensated BF16 path on a large operator
        {"name": "krylov_bf16", "kind": "krylov", "n": 4096, "m": 30, "precision": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges, odd sizes among them."""
    kind = rng.choice(["rta", "rta", "rta_poly", "rta_spectral", "rta_batch", "rta_grad", "fit", "bert", "bert",
                       "bert_heated", "krylov", "krylov"])
    if kind == "krylov":
        prec = rng.choice(["fp64", "fp32", "bf16"])
        return {"kind": kind, "n": _log_int(rng, 257, 2500 if prec == "fp64" else 3500), "m": rng.randint(20, 30),
                "precision": prec}
    if kind == "bert":
        return {"kind": kind, "modes": _log_int(rng, 300, 2000), "particles": _log_int(rng, 30000, 1000000),
                "bins": rng.randint(11, 60), "replicas": rng.choice([1, 1, 2, 3]), "steps": rng.randint(30, 120)}
    if kind == "bert_heated":
        return {"kind": kind, "modes": _log_int(rng, 200, 2000), "particles": _log_int(rng, 30000, 300000),
                "bins": rng.randint(11, 60), "steps": rng.randint(30, 80)}
    case = {"kind": kind, "modes": 2 * _log_int(rng, 150, 1500) if kind in ("rta_grad", "fit")
            else _log_int(rng, 300, 3000),
            "length": float(rng.randint(150, 1000)), "bins": rng.randint(15, 100),
            "maxtime": float(rng.randint(500, 3000)), "steps": rng.randint(25, 150)}
    if kind == "rta_batch":
        case.update(runs=rng.randint(3, 16), min_particles=_log_int(rng, 5000, 30000),
                    max_particles=_log_int(rng, 50000, 800000))
        return case
    case["particles"] = _log_int(rng, 2000, 1000000) if kind in ("rta", "rta_grad") else _log_int(rng, 5000, 200000)
    case["width"] = float(rng.randint(40, 300))
    if kind == "rta_poly":
        case.update(bins=2 * rng.randint(7, 25) + 1, width=float(rng.randint(60, 120)))
        case["length"] = 10.0 * case["bins"]
    elif kind == "rta_spectral":
        case.update(locations=rng.randint(1, 4), ticks=rng.randint(50, 150))
    elif kind in ("rta_grad", "fit"):
        case.update(p_top=round(rng.uniform(0.1, 0.9), 3), p_bottom=round(rng.uniform(0.1, 0.9), 3))
        if kind == "fit":
            case["bins"], case["steps"] = rng.randint(15, 40), rng.randint(20, 50)
        else:
            # five FP32 arrays of bins x time bins share a workgroup's 160 KB
            case["steps"] = min(case["steps"], 8000 // case["bins"])
    return case


# ---- inputs ----

def _modes(mat):
    return bte.ModeTable(_ctx(), mat["omega"], mat["vx"], mat["vy"], mat["w"], mat["V"], mat["lattz"])


def _ribbon_geom(case, width, T=300.0):
    rect, kind, teq, _ = bte.workloads.ribbon(case["length"], width, case["bins"], T,
                                              reservoirs=(T + 0.5, T - 0.5))
    return bte.Geometry(_ctx(), rect, kind, teq)


def _zigzag(case):
    """Quadrilateral cells along x with slanted shared sides and a zigzag top
    edge, and a reservoir rectangle at each end."""
    n, L, H = case["bins"], case["length"], case["width"]
    dx = L / n
    x = np.linspace(0.0, L, n + 1)
    s = 0.2 * dx * (-1.0) ** np.arange(n + 1)
    s[0] = s[-1] = 0.0
    h = H + 0.1 * H * (-1.0) ** np.arange(n + 1)
    polys = [np.array([[x[i], 0.0], [x[i + 1], 0.0], [x[i + 1] + s[i + 1], h[i + 1]], [x[i] + s[i], h[i]]])
             for i in range(n)]
    polys.append(np.array([[-dx, 0.0], [0.0, 0.0], [0.0, h[0]], [-dx, h[0]]]))
    polys.append(np.array([[L, 0.0], [L + dx, 0.0], [L + dx, h[-1]], [L, h[-1]]]))
    kind = np.array([0] * n + [1, 1], np.int32)
    teq = np.array([300.0] * n + [300.5, 299.5])
    return bte.Geometry(_ctx(), None, kind, teq, polys=polys)


def _heated_bar(nbins, dx=10.0, width=60.0):
    """A bar of nbins boxes at 300 K, heated by a 301 K reservoir at its left
    end, a 300 K one at the right, periodic in y through ghost boxes."""
    L = nbins * dx
    rect = [[k * dx, (k + 1) * dx, 0.0, width] for k in range(nbins)]
    rect += [[0.0, L, -2.0, 0.0], [0.0, L, width, width + 2.0]]
    rect += [[-dx, 0.0, 0.0, width], [L, L + dx, 0.0, width]]
    kind = np.array([0] * nbins + [2, 2, 1, 1], np.int32)
    teq = np.array([300.0] * (nbins + 2) + [301.0, 300.0])
    periodic = {nbins: (nbins + 1, 0.0, width), nbins + 1: (nbins, 0.0, -width)}
    return bte.Geometry(_ctx(), np.array(rect), kind, teq, periodic=periodic)


def _operator(n, seed):
    """A collision operator B = -Omega of n modes: symmetric random couplings
    of 5 % density between all pairs, scaled so that columns sum to zero, the
    heat capacities are its null vector and the rates spread over 1 ps - 1 ns."""
    r = np.random.default_rng(seed)
    om = 2.0 * np.pi * r.uniform(0.1, 15.0, n)
    w = 10.0 ** -r.uniform(0.0, 3.0, n)
    x = 0.5e12 * 1.054571726e-34 * om / (1.3806488e-23 * 300.0)
    c = (x / np.sinh(x)) ** 2
    g = c * w
    S = np.triu(r.random((n, n), dtype=np.float32).astype(np.float64), 1)
    S[S > 0.05] = 0.0  # what stays is uniform in (0, 0.05): density 5 %
    S += S.T
    S *= (g / (g.sum() * 0.05 * 0.025))[:, None]
    S *= g[None, :]
    rows = S.sum(axis=1)
    S[np.arange(n), np.arange(n)] -= rows
    return np.asfortranarray(S / c[None, :])


DT = 5.0  # ps, the propagator's time step


def _sigma(case):
    """Broadening of the diffuse bounce [rad/ps]: the benchmarks' 0.25, wider
    for small mode tables so that every mode has partners."""
    return 0.25 if case["modes"] >= 2000 else 1.0


def prepare(case, seed):
    kind = case["kind"]
    s = int(seed) % 100000 + 1
    W = bte.workloads
    if kind == "krylov":
        return {"case": case, "B": _operator(case["n"], s)}
    if kind == "bert":
        mat, B = W.config1_inputs(case["modes"], seed=s)
        P, _ = bte.build_P(_ctx(), B, DT, m=30, precision="fp64")
        c = W.config1(nsteps=case["steps"], dt=DT, nparticles=case["particles"], nbins=case["bins"], seed=s,
                      replicas=case["replicas"])
        geom = bte.Geometry(_ctx(), c["rect"], c["kind"], c["Teq"], c["Tinit"])
        run = bte.BertRun(_ctx(), _modes(mat), geom, bte.Propagator(_ctx(), P), thickness=c["thickness"],
                          dt=c["dt"], maxtime=c["maxtime"], max_steps=c["max_steps"], Efactor=c["Efactor"],
                          Tmax=c["Tmax"], Tmin=c["Tmin"], seed=s)
        return {"case": case, "run": run}
    mat = W.material(case["modes"], seed=s, mirror=kind in ("rta_grad", "fit"))
    modes = _modes(mat)
    if kind == "bert_heated":
        geom = _heated_bar(case["bins"])
        run = bte.BertRun(_ctx(), modes, geom, None, thickness=1.0, dt=2.0, maxtime=2.0 * (case["steps"] - 1),
                          max_steps=case["steps"], rta=True, Efactor=case["particles"] // case["bins"] + 1,
                          Tmax=301.0, Tmin=300.0, seed=s)
        return {"case": case, "run": run}
    kw = dict(thickness=1.0, dt=case["maxtime"] / case["steps"], maxtime=case["maxtime"])
    if kind in ("rta", "rta_poly", "rta_spectral"):
        geom = _zigzag(case) if kind == "rta_poly" else _ribbon_geom(case, case["width"])
        run = bte.RtaRun(_ctx(), modes, geom, T0=300.0, nparticles=case["particles"], seed=s, sigma_bounce=_sigma(case), **kw)
        if kind == "rta_spectral":
            k = case["locations"]
            run.spectral([int((i + 0.5) * case["bins"] / k) for i in range(k)], case["ticks"], np.full(mat["n"], 1.0))
        return {"case": case, "run": run}
    if kind == "rta_batch":
        n = case["runs"]
        widths = np.geomspace(50.0, 2000.0, n)
        temps = np.linspace(100.0, 500.0, n)
        counts = np.random.default_rng(s).permutation(
            np.geomspace(case["min_particles"], case["max_particles"], n)).astype(int)
        runs = [dict(geom=_ribbon_geom(case, float(widths[i]), float(temps[i])), T0=float(temps[i]),
                     nparticles=int(counts[i]), seed=1000 * s + i, wscale=float(temps[i]) / 300.0) for i in range(n)]
        return {"case": case, "run": bte.RtaBatch(_ctx(), modes, runs, sigma_bounce=_sigma(case), tally="fp64-lds-runs", **kw)}
    geom = _ribbon_geom(case, case["width"])
    if kind == "rta_grad":
        spec = (0.0, case["p_bottom"], case["p_top"], 0.0)  # left, bottom, top, right
        runs = [dict(geom=geom, T0=300.0, nparticles=case["particles"], seed=s, specularity=spec, grad=True)]
        return {"case": case, "run": bte.RtaBatch(_ctx(), modes, runs, sigma_bounce=_sigma(case), tally="fp32-lds", **kw)}
    if kind == "fit":
        model = _autograd.SpecularityModel(bte, _ctx(), modes, geom, T0=300.0, nparticles=case["particles"],
                                           seed=s, sigma_bounce=_sigma(case), **kw)
        p = torch.tensor([0.0, case["p_bottom"], case["p_top"], 0.0], dtype=torch.float64, device="cuda")
        target = 300.0 + torch.linspace(0.4, -0.4, case["bins"] + 2, dtype=torch.float64, device="cuda")
        return {"case": case, "model": model, "p": p, "target": target}
    raise ValueError("unknown kind %r" % kind)


# ---- one pass ----

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "krylov":
        P, rep = bte.build_P(_ctx(), state["B"], DT, m=case["m"], precision=case["precision"])
        return {"P": P, "breakdowns": rep["breakdowns"]}
    if kind in ("bert", "bert_heated"):
        o = state["run"].execute()
        return {k: o[k] for k in ("props", "npart", "pending", "nsteps", "particle_steps",
                                  "step_kernel_particle_steps", "max_particles")}
    if kind == "rta_batch":
        outs, rep = state["run"].execute()
        return {"T": np.stack([o["T"] for o in outs]), "jx": np.stack([o["jx"] for o in outs]),
                "jy": np.stack([o["jy"] for o in outs]), "events": rep["events"], "crossings": rep["crossings"]}
    if kind == "rta_grad":
        (o,), rep = state["run"].execute(grad=True)
        return {"T": o["T"], "jx": o["jx"], "jy": o["jy"], "dTdp": o["dTdp"], "events": rep["events"],
                "crossings": rep["crossings"]}
    if kind == "fit":
        p = state["p"].clone().requires_grad_(True)
        T = state["model"](p)
        loss = (T[-1] - state["target"]).square().sum()
        loss.backward()
        return {"T": T.detach(), "loss": loss.detach(), "grad": p.grad}
    o = state["run"].execute()
    out = {k: o[k] for k in ("T", "jx", "jy", "events", "crossings")}
    if kind == "rta_spectral":
        out["spectral"] = [{k: d[k] for k in ("dT", "jx", "jy", "fd")} for d in o["spectral"]]
    return out


def exact(case, seed):
    if case["kind"] != "krylov":
        return None
    B = torch.from_numpy(_operator(case["n"], int(seed) % 100000 + 1)).to("cuda")
    P = torch.linalg.matrix_exp(DT * B)
    P += (1.0 - P.sum(dim=0, keepdim=True)) / case["n"]
    return {"P": P.cpu().numpy(), "breakdowns": None}


# ---- what a pass cannot do without ----

def _rta_flights(particles, length, maxtime, bins, wscale=1.0):
    """Flights and box crossings of a run. A particle stays L / (2 <vx+>) on
    average (the mean chord of the ribbon, <vx+> = 4.25 / pi nm/ps for this
    material), scatters at the mean rate 0.145 / ps and crosses a side every
    dx / <|vx|>."""
    vx = 4.25 / math.pi
    t = min(maxtime, length / (2.0 * vx))
    return particles * t * 0.145 * wscale, particles * t * 2.0 * vx * bins / length


# FP64 operations of a flight (logarithm, end point, exit test, tally) and of
# a crossing (exit time, end point, tally)
FLIGHT_FLOPS, CROSSING_FLOPS = 60.0, 30.0


def work(case):
    kind = case["kind"]
    if kind == "krylov":
        n = case["n"]
        parts = 3 if case["precision"] == "bf16" else 1
        return {"bytes": 16.0 * n * n, "flops": parts * 2.0 * (case["m"] - 1) * float(n) ** 3}
    if kind in ("bert", "bert_heated"):
        # a particle-step: 32 B of state in and out and one 8-B table entry
        ps = case["particles"] * case.get("replicas", 1) * case["steps"] * (0.5 if kind == "bert_heated" else 1.0)
        return {"bytes": 72.0 * ps, "flops": 60.0 * ps}
    cells = (case["bins"] + 2) * case["steps"]
    if kind == "rta_batch":
        n = case["runs"]
        counts = np.geomspace(case["min_particles"], case["max_particles"], n)
        ev, cr = _rta_flights(float(counts.sum()), case["length"], case["maxtime"], case["bins"])
        return {"bytes": 24.0 * n * cells + 120.0 * case["modes"] * n,
                "flops": FLIGHT_FLOPS * ev + CROSSING_FLOPS * cr}
    ev, cr = _rta_flights(case["particles"], case["length"], case["maxtime"], case["bins"])
    arrays = 7 if kind in ("rta_grad", "fit") else 3
    out = {"bytes": 8.0 * arrays * cells + 120.0 * case["modes"], "flops": FLIGHT_FLOPS * ev + CROSSING_FLOPS * cr}
    if kind == "rta_spectral":
        cols = 3 * case["ticks"] + 1
        out["bytes"] += 8.0 * cols * (case["locations"] * case["steps"] + case["modes"])
        out["flops"] += 2.0 * case["locations"] * case["steps"] * case["modes"] * cols
    return out
