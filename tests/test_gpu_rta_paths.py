"""The history kernels' routes: boxes, polygon sides and time grid in LDS or,
past 20 KB, in global memory; waves with one lane up to full waves; histories
that change waves once the ids have run out. A run's histories depend on its
seed and particle ids only, so every route gives the same event and crossing
counts and, up to the order of the FP64 sums, the same T, jx and jy (1e-10 of
the largest magnitude, as in the tally-mode tests)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KW = dict(thickness=1.0, dt=10.0, maxtime=400.0, sigma_bounce=2.0)


def _modes(pkg, ctx, n=300, mirror=True):
    m = pkg.workloads.material(n, seed=3, mirror=mirror)
    return pkg.ModeTable(ctx, m["omega"], m["vx"], m["vy"], m["w"], m["V"], m["lattz"])


def _ribbon(pkg, ctx, nb, width=40.0, dx=10.0, poly=False):
    rect, kind, teq, _ = pkg.workloads.ribbon(nb * dx, width, nb, 300.0, reservoirs=(300.5, 299.5))
    polys = None
    if poly:
        # slanted shared sides: neighbours meet along x = k dx +- 2 (bottom to top)
        polys = [np.array([[r[0], r[2]], [r[1], r[2]], [r[1], r[3]], [r[0], r[3]]]) for r in rect]
        for k in range(nb):
            if k > 0:
                polys[k][3, 0] += 2.0
            if k < nb - 1:
                polys[k][2, 0] += 2.0
    return pkg.Geometry(ctx, rect, kind, teq, polys=polys)


def _same(a, b):
    for key, off in (("T", 300.0), ("jx", 0.0), ("jy", 0.0)):
        scale = np.abs(b[key] - off).max()
        np.testing.assert_allclose(a[key] - off, b[key] - off, rtol=0, atol=1e-10 * scale)


# in LDS: 80 B a box, 56 B a polygon side, 8 B a time step, at most 20480 B;
# 250 rectangles or 70 quadrilaterals are the last that fit next to 41 steps
@pytest.mark.parametrize("tally", ["fp64", "fp64-lds", "fp64-lds-runs", "fp32-lds"])
@pytest.mark.parametrize("poly,nb", [(False, 8), (False, 249), (False, 251), (True, 9), (True, 75)])
def test_geometry_in_lds_and_in_global_memory(pkg, ctx, tally, poly, nb):
    """One ribbon alone (its geometry in LDS while it fits) and beside a second
    ribbon that takes the batch past the LDS limit."""
    modes = _modes(pkg, ctx)
    geom, other = _ribbon(pkg, ctx, nb, poly=poly), _ribbon(pkg, ctx, 260, poly=poly)
    run = dict(geom=geom, T0=300.0, nparticles=30000, seed=5)
    kw = dict(KW)
    if tally == "fp32-lds":
        kw.update(dt=80.0)  # every time bin of every box has to fit in LDS
    tol = 1e-4 if tally == "fp32-lds" else 1e-10
    ref_b = pkg.RtaBatch(ctx, modes, [run], **kw)
    (ref,), rep = ref_b.execute()
    ref_b.close()
    one = pkg.RtaBatch(ctx, modes, [run], tally=tally, **kw)
    (got,), grep = one.execute()
    one.close()
    assert (grep["events"], grep["crossings"]) == (rep["events"], rep["crossings"])
    both = [got]
    if tally != "fp32-lds" or not poly:
        two = pkg.RtaBatch(ctx, modes, [run, dict(geom=other, T0=300.0, nparticles=100, seed=6)], tally=tally, **kw)
        res, _ = two.execute()
        two.close()
        both.append(res[0])
    for g in both:
        for key, off in (("T", 300.0), ("jx", 0.0), ("jy", 0.0)):
            scale = np.abs(ref[key] - off).max()
            assert scale > 0
            np.testing.assert_allclose(g[key] - off, ref[key] - off, rtol=0, atol=tol * scale)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 3071, 3073, 50000, 200001])
def test_particle_counts_around_the_lanes_of_the_gpu(pkg, ctx, n):
    """From one history to more than one per lane: waves with a single lane,
    partly filled waves and refills, under every tally mode."""
    modes = _modes(pkg, ctx)
    run = dict(geom=_ribbon(pkg, ctx, 12), T0=300.0, nparticles=n, seed=9, specularity=(0.0, 0.5, 1.0, 0.0))
    out = {}
    for tally in ("fp64", "fp64-lds", "fp64-lds-runs", "fp32-lds"):
        b = pkg.RtaBatch(ctx, modes, [run], tally=tally, **KW)
        (out[tally],), rep = b.execute()
        b.close()
        out[tally]["counts"] = (rep["events"], rep["crossings"])
    for tally in ("fp64-lds", "fp64-lds-runs"):
        assert out[tally]["counts"] == out["fp64"]["counts"]
        _same(out[tally], out["fp64"])
    assert out["fp32-lds"]["counts"] == out["fp64"]["counts"]


def test_scores_move_with_their_histories(pkg, ctx):
    """dT/dp in FP64 tallies: the ribbon alone (LDS geometry) and in a batch
    past the LDS limit (global geometry)."""
    modes = _modes(pkg, ctx)
    run = dict(geom=_ribbon(pkg, ctx, 20), T0=300.0, nparticles=60000, seed=11, specularity=(0.0, 0.4, 0.6, 0.0),
               grad=True)
    a = pkg.RtaBatch(ctx, modes, [run], **KW)
    (ra,), rep_a = a.execute(grad=True)
    a.close()
    b = pkg.RtaBatch(ctx, modes, [run, dict(geom=_ribbon(pkg, ctx, 260), T0=300.0, nparticles=100, seed=6)], **KW)
    rb, _ = b.execute(grad=True)
    b.close()
    _same(rb[0], ra)
    scale = np.abs(ra["dTdp"]).max()
    assert scale > 0
    np.testing.assert_allclose(rb[0]["dTdp"], ra["dTdp"], rtol=0, atol=1e-10 * scale)


@pytest.mark.parametrize("nruns", [1, 3, 300])
def test_runs_shared_among_workgroups(pkg, ctx, nruns):
    """Tally mode 3 with one run for all workgroups, a few uneven ones, and
    more runs than workgroups (those without one are picked up later)."""
    modes = _modes(pkg, ctx, n=100)
    geom = _ribbon(pkg, ctx, 6)
    counts = [int(c) for c in (np.geomspace(60000, 900, nruns) if nruns < 10 else 20 + 37 * (np.arange(nruns) % 11))]
    runs = [dict(geom=geom, T0=300.0, nparticles=c, seed=40 + k, wscale=0.5 + k / nruns)
            for k, c in enumerate(counts)]
    ref_b = pkg.RtaBatch(ctx, modes, runs, **KW)
    ref, rep = ref_b.execute()
    ref_b.close()
    b = pkg.RtaBatch(ctx, modes, runs, tally="fp64-lds-runs", **KW)
    for _ in range(2):
        got, grep = b.execute()
        assert (grep["events"], grep["crossings"]) == (rep["events"], rep["crossings"])
        for g, r in zip(got, ref):
            _same(g, r)
    b.close()


@pytest.mark.parametrize("tally", ["fp64", "fp64-lds-runs"])
def test_modes_without_scattering(pkg, ctx, tally):
    """A rate below the smallest normal number, whose reciprocal overflows,
    draws flights longer than any run: they end at maxtime, as with a rate so
    small that no flight ends before it. (Rates of 0 are refused.)"""
    m = pkg.workloads.material(200, seed=3, mirror=True)
    geom = _ribbon(pkg, ctx, 12)
    out = []
    for w in (1e-30, 1e-310):
        modes = pkg.ModeTable(ctx, m["omega"], m["vx"], m["vy"], np.full(200, w), m["V"], m["lattz"])
        b = pkg.RtaBatch(ctx, modes, [dict(geom=geom, T0=300.0, nparticles=5000, seed=2)], tally=tally, **KW)
        (r,), rep = b.execute()
        b.close()
        out.append((r, rep["events"], rep["crossings"]))
    assert out[0][2] > 5000
    for r, ev, cr in out[1:]:
        assert (ev, cr) == out[0][1:]
        _same(r, out[0][0])


# events and crossings with the tables made on the host, one mode after the other
@pytest.mark.parametrize("n,sigma,own,want", [(300, 2.0, False, (60479, 21616)), (300, 2.0, True, (61429, 22044)),
                                              (2200, 1e3, False, (68168, 24881))])
def test_lambert_tables(pkg, ctx, n, sigma, own, want):
    """The diffuse-bounce tables of every mode and side normal, with one width
    or one per mode; windows of all 2200 modes make more entries than one pass takes."""
    m = pkg.workloads.material(n, seed=5)
    rect, kind, teq, _ = pkg.workloads.ribbon(60.0, 5.0, 6, 300.0, reservoirs=(302.0, 300.0))
    modes = pkg.ModeTable(ctx, m["omega"], m["vx"], m["vy"], m["w"], m["V"], m["lattz"])
    if own:
        modes.set_sigma(np.random.default_rng(1).uniform(0.5, 3.0, n))
    b = pkg.RtaBatch(ctx, modes, [dict(geom=pkg.Geometry(ctx, rect, kind, teq), T0=300.0, nparticles=4000, seed=2)],
                     thickness=1.0, dt=10.0, maxtime=400.0, sigma_bounce=sigma)
    _, rep = b.execute()
    b.close()
    assert (rep["events"], rep["crossings"]) == want


def test_lambert_window_without_partner(pkg, ctx):
    """A width so small that a mode's window holds the mode alone: the first
    one that can reach a side is named."""
    m = pkg.workloads.material(200, seed=5)
    modes = pkg.ModeTable(ctx, m["omega"], m["vx"], m["vy"], m["w"], m["V"], m["lattz"])
    with pytest.raises(pkg.BteError, match="mode 0 has no diffuse partner within the Lambert window"):
        pkg.RtaBatch(ctx, modes, [dict(geom=_ribbon(pkg, ctx, 6), T0=300.0, nparticles=100, seed=2)],
                     **dict(KW, sigma_bounce=1e-9))


@pytest.mark.parametrize("nb", [8, 249])
def test_fp64_lds_tallies_launch_what_runs_at_a_time(pkg, ctx, nb):
    """One 768-thread workgroup per CU, whether one tally block or two fit its
    LDS (the device atomics' launch is eight 256-thread workgroups per CU)."""
    run = dict(geom=_ribbon(pkg, ctx, nb), T0=300.0, nparticles=30000, seed=5)
    reps = []
    for tally in ("fp64", "fp64-lds"):
        b = pkg.RtaBatch(ctx, _modes(pkg, ctx), [run], tally=tally, **KW)
        reps.append(b.execute()[1])
        b.close()
    assert reps[0]["block"] == 256 and reps[1]["block"] == 768
    assert reps[1]["blocks"] == reps[0]["blocks"] // 8
    assert reps[1]["events"] == reps[0]["events"]


def test_diffuse_partners_without_broadening_or_frequency(pkg, ctx):
    """Three of eight modes at zero frequency and with a per-mode broadening
    of 0 (a quarter of the modes: the broadening's floor is 0 too). They are
    nobody's diffuse partner, so the width of their pairs, 0, enters no
    table, and the other five scatter at the walls as without them."""
    omega = np.array([0.0, 0.0, 0.0, 10.0, 10.0, 10.1, 10.1, 10.2])
    v = np.array([[1.0, 0.5], [-1.0, 0.5], [0.5, -1.0], [2.0, 2.0], [-2.0, -2.0], [2.0, -2.0], [-2.0, 2.0], [1.0, 1.5]])
    modes = pkg.ModeTable(ctx, omega, v[:, 0], v[:, 1], np.full(8, 0.1), 1.0, 1.0)
    modes.set_sigma(np.array([0.0] * 3 + [0.5] * 5))
    five = pkg.ModeTable(ctx, omega[3:], v[3:, 0], v[3:, 1], np.full(5, 0.1), 1.0, 1.0)
    five.set_sigma(np.full(5, 0.5))
    out = []
    for m in (modes, five):
        run = pkg.RtaRun(ctx, m, _ribbon(pkg, ctx, 4, width=10.0), thickness=1.0, T0=300.0, dt=10.0, maxtime=100.0,
                         nparticles=2000, seed=3)
        out.append(run.execute())
        run.close()
    for o in out:
        assert o["events"] > 2000 and np.isfinite(o["T"]).all()
    # a history has a few tens of events at most (10 scatterings and 20 walls
    # on average for one that stays), so their number varies by less than its mean
    assert abs(out[0]["events"] / out[1]["events"] - 1.0) < 5.0 * np.sqrt(2.0 / 2000)
