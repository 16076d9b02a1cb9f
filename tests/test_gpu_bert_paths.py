"""Routes of the beRTAMC2D particle kernels on geometries around the LDS
limits: boxes in LDS (at most 614, 80 bytes each) or in global memory, the
velocity tables beside them or not, wall counters in LDS (at most 2048 sides) or
global. The histories follow the particle ids, so the two launch shapes agree
exactly in their particle counts and, up to the order of the FP64 sums, in
the box sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,rows,n", [(5, 1, 60), (307, 2, 60), (310, 2, 60), (40, 3, 4000), (500, 1, 3600)])
def test_launch_shapes_agree(pkg, ctx, nb, rows, n):
    """rows of nb boxes, stacked in y so that corners are shared by four boxes"""
    W = pkg.workloads
    mat = W.material(n, seed=5)
    rect = [[k * 10.0, (k + 1) * 10.0, r * 12.0, (r + 1) * 12.0] for r in range(rows) for k in range(nb)]
    kind = np.zeros(len(rect), np.int32)
    teq = np.full(len(rect), 300.0)
    tin = teq.copy()
    tin[: min(3, nb)] = 304.0
    modes = pkg.ModeTable(ctx, mat["omega"], mat["vx"], mat["vy"], mat["w"], mat["V"], mat["lattz"])
    geom = pkg.Geometry(ctx, np.array(rect), kind, teq, tin)
    kw = dict(thickness=1.0, dt=4.0, maxtime=36.0, max_steps=10, rta=True, Efactor=20000, Tmax=304.0, Tmin=300.0,
              seed=3)
    out = []
    for shape in (0, 1):
        b = pkg.BertRun(ctx, modes, geom, None, step_shape=shape, **kw)
        out.append(b.execute())
        b.close()
    a, c = out
    assert np.array_equal(a["npart"], c["npart"]) and np.array_equal(a["pending"], c["pending"])
    assert (a["npart"] + a["pending"] == a["npart"][0]).all() and a["npart"][0] > 0
    scale = np.abs(c["props"]).max(axis=(0, 1))
    np.testing.assert_allclose(a["props"] / scale, c["props"] / scale, rtol=0, atol=1e-10)


def _periodic_bar(nb, extra, width=30.0, dx=10.0):
    """nb boxes periodic in y between a 302 K and a 300 K reservoir, and
    `extra` bars of the same kind without a temperature difference far away"""
    rect, kind, teq, per = [], [], [], {}
    for e in range(1 + extra):
        y0, L, b0 = 1000.0 * e, nb * dx, len(rect)
        rect += [[k * dx, (k + 1) * dx, y0, y0 + width] for k in range(nb)]
        rect += [[0.0, L, y0 - 2.0, y0], [0.0, L, y0 + width, y0 + width + 2.0]]
        rect += [[-dx, 0.0, y0, y0 + width], [L, L + dx, y0, y0 + width]]
        kind += [0] * nb + [2, 2, 1, 1]
        teq += [300.0] * (nb + 2) + [302.0 if e == 0 else 300.0, 300.0]
        per.update({b0 + nb: (b0 + nb + 1, 0.0, width), b0 + nb + 1: (b0 + nb, 0.0, -width)})
    return np.array(rect), np.array(kind, np.int32), np.array(teq), per


@pytest.mark.parametrize("nb,extra", [(12, 20), (70, 3), (150, 1)])
def test_periodic_tables_in_lds_and_in_global_memory(pkg, ctx, nb, extra):
    """A bar alone (its boxes and periodic tables in LDS; past 64 contacts the
    search takes several rounds) and with others that push the tables past
    48 KB: the bar's histories are the same."""
    W = pkg.workloads
    mat = W.material(80, seed=5)
    modes = pkg.ModeTable(ctx, mat["omega"], mat["vx"], mat["vy"], mat["w"], mat["V"], mat["lattz"])
    kw = dict(thickness=1.0, dt=4.0, maxtime=76.0, max_steps=20, rta=True, seed=3)
    out = []
    Ed = -1.0
    for e in (0, extra):
        rect, kind, teq, per = _periodic_bar(nb, e)
        geom = pkg.Geometry(ctx, rect, kind, teq, periodic=per)
        b = pkg.BertRun(ctx, modes, geom, None, Ed=Ed, Efactor=400, Tmax=302.0, Tmin=300.0, **kw)
        out.append(b.execute())
        Ed = out[0]["Eeff"]
        b.close()
    a, c = out
    assert np.array_equal(a["npart"], c["npart"]) and a["npart"][-1] > 1000
    scale = np.abs(a["props"]).max(axis=(0, 1))
    np.testing.assert_allclose(c["props"][:, :nb] / scale, a["props"][:, :nb] / scale, rtol=0, atol=1e-10)


@pytest.mark.parametrize("pc", [1, 2, 4])
@pytest.mark.parametrize("steps", [1, 2, 9])
def test_properties_of_each_step(pkg, ctx, pc, steps):
    """A step's properties, particle count and pending wall hits are taken
    while the next step runs (the last step's afterwards), from box sums or,
    where it cancels, the histogram. The frames of a second run hold that
    histogram after each step: its net sum times the energy per particle and
    volume is the first property, and its net counts those left where the
    step cancels. A third run, which its callback stops, has the same rows up
    to there."""
    W = pkg.workloads
    mat = W.material(60, seed=5)
    rect, kind, teq, _ = W.ribbon(60.0, 5.0, 6, 300.0, reservoirs=(302.0, 300.0))  # narrow: emitted particles reach the other side
    modes = pkg.ModeTable(ctx, mat["omega"], mat["vx"], mat["vy"], mat["w"], mat["V"], mat["lattz"])
    geom = pkg.Geometry(ctx, rect, kind, teq)
    kw = dict(thickness=1.0, dt=4.0, maxtime=4.0 * (steps - 1), max_steps=steps, rta=True, Efactor=4000, Tmax=302.0,
              Tmin=300.0, seed=3, pcancel_each=pc)

    def run(cb=None):
        b = pkg.BertRun(ctx, modes, geom, None, **kw)
        r = b.execute() if cb is None else b.execute(cb)
        b.close()
        return r

    frames = []
    a = run()
    c = run(lambda s, t, e, H: frames.append((e, H)) and False)
    assert len(frames) == steps == len(a["npart"]) - 1
    for key in ("npart", "pending"):
        assert np.array_equal(a[key], c[key]), key
    np.testing.assert_allclose(a["props"], c["props"], rtol=1e-10, atol=1e-10 * np.abs(a["props"]).max())
    area = (rect[:, 1] - rect[:, 0]) * (rect[:, 3] - rect[:, 2])
    reg = np.asarray(kind) == 0
    assert a["npart"][-1] > 0 and (steps < 9 or a["pending"][1:].any())
    for s, (e, H) in enumerate(frames):
        want = e / area * 1.0e27 * H.sum(1)
        np.testing.assert_allclose(a["props"][s + 1, reg, 0], want[reg], rtol=1e-12, atol=0)
        if s % pc == 0:
            assert a["npart"][s + 1] == np.abs(H[reg]).sum()
    stop = run(lambda s, t, e, H: s == steps // 2)
    assert np.array_equal(stop["npart"][:steps // 2 + 2], a["npart"][:steps // 2 + 2])
    assert np.array_equal(stop["pending"][:steps // 2 + 2], a["pending"][:steps // 2 + 2])


@pytest.mark.parametrize("nb", [1, 3, 8, 33])
def test_wall_workgroups_cover_every_side(pkg, ctx, nb):
    """Sides are dealt to the wall workgroups by fours, in polygon geometries
    of 4 nb + 3 sides (one box a triangle, so that their number is no multiple
    of four) as in nb + 1 rectangles: with adiabatic walls all around, every
    particle that hits one comes out of it again, none is lost over the run."""
    W = pkg.workloads
    mat = W.material(60, seed=5)
    modes = pkg.ModeTable(ctx, mat["omega"], mat["vx"], mat["vy"], mat["w"], mat["V"], mat["lattz"])
    for tri in (False, True):
        rect = np.array([[k * 10.0, (k + 1) * 10.0, 0.0, 12.0] for k in range(nb + 1)])
        polys = [np.array([[r[0], r[2]], [r[1], r[2]], [r[1], r[3]], [r[0], r[3]]]) for r in rect]
        if tri:
            x = nb * 10.0
            polys[nb] = np.array([[x, 0.0], [x + 9.0, 6.0], [x, 12.0]])
        teq = np.full(nb + 1, 300.0)
        tin = teq.copy()
        tin[0] = 304.0
        geom = pkg.Geometry(ctx, rect, np.zeros(nb + 1, np.int32), teq, tin, polys=polys if tri else None)
        b = pkg.BertRun(ctx, modes, geom, None, thickness=1.0, dt=4.0, maxtime=36.0, max_steps=10, rta=True,
                        Efactor=20000, Tmax=304.0, Tmin=300.0, seed=3)
        r = b.execute()
        b.close()
        assert r["npart"][0] > 5000
        assert (r["npart"] + r["pending"] == r["npart"][0]).all(), (tri, r["npart"], r["pending"])


@pytest.mark.parametrize("nb,seed", [(2, 1), (6, 1), (6, 2)])
def test_wall_hits_that_cancel(pkg, ctx, nb, seed):
    """Few particles of both signs between adiabatic walls 5 nm apart: the
    hits of a side from the step and from the emission before often cancel.
    Every step keeps the signed particle count: those in the boxes (the first
    property is their net count times the energy per particle and volume) and
    the hits that wait for their emission."""
    W = pkg.workloads
    mat = W.material(60, seed=5)
    L = 10.0
    rect = np.array([[k * L, (k + 1) * L, r * 8.0, r * 8.0 + 5.0] for r in range(2) for k in range(nb)])
    teq = np.full(2 * nb, 300.0)
    tin = np.repeat([303.0, 297.0], nb)
    tin[1::2] = 600.0 - tin[1::2]  # hot and cold boxes in turn, opposite in the second row
    modes = pkg.ModeTable(ctx, mat["omega"], mat["vx"], mat["vy"], mat["w"], mat["V"], mat["lattz"])
    geom = pkg.Geometry(ctx, rect, np.zeros(2 * nb, np.int32), teq, tin)
    b = pkg.BertRun(ctx, modes, geom, None, thickness=1.0, dt=4.0, maxtime=4.0 * 399, max_steps=400, rta=True,
                    Efactor=40, Tmax=303.0, Tmin=297.0, seed=seed, pcancel_each=1000)
    r = b.execute()
    b.close()
    net = r["props"][:, :, 0].sum(1) * (L * 5.0) / (r["Eeff"] * 1.0e27) + r["pending"]
    assert r["npart"][0] > 20 and r["pending"].any()
    np.testing.assert_allclose(net, round(net[0]), rtol=0, atol=1e-6)


def test_a_given_capacity_holds_with_a_large_source(pkg, ctx):
    """A source of about 1e5 particles per step beside 2e6 initial ones, in a
    given capacity: with a source segment for every 1024 particles (98 beside
    256 of the step kernel and 256 of the emission) a segment of 0.95 of the
    step workgroups' share of the initial particles is enough, as 15 percent
    of them leave or wait at a wall in the first step; with one for every 256
    (256 at most) it would be 0.75. The histories are those of the automatic
    capacity."""
    W = pkg.workloads
    mat = W.material(60, seed=5)
    rect, kind, teq, _ = W.ribbon(100.0, 200.0, 5, 300.0, reservoirs=(302.0, 300.0))
    tin = np.where(np.asarray(kind) == 0, 302.0, teq)
    modes = pkg.ModeTable(ctx, mat["omega"], mat["vx"], mat["vy"], mat["w"], mat["V"], mat["lattz"])
    geom = pkg.Geometry(ctx, rect, kind, teq, tin)

    def run(**kw):
        b = pkg.BertRun(ctx, modes, geom, None, thickness=1.0, dt=4.0, maxtime=8.0, rta=True, Efactor=400000,
                        Tmax=302.0, Tmin=300.0, seed=3, pcancel_each=1000, **kw)
        r = b.execute()
        b.close()
        return r

    a = run()
    n0 = int(a["npart"][0])
    assert n0 > 1900000 and a["npart"].max() == n0 and a["step_threads"] == 1024
    c = run(capacity=int(0.95 * n0 / 256 * (256 + 256 + 98)))
    assert np.array_equal(a["npart"], c["npart"]) and np.array_equal(a["pending"], c["pending"])


@pytest.mark.parametrize("pc,steps,timed", [(4, 16, 4), (4, 15, 3), (4, 100, 7), (1, 9, 3), (2, 8, 2), (6, 36, 6)])
def test_timed_steps_reach_every_place_of_the_cycle(pkg, ctx, pc, steps, timed):
    """One launch in every fourth cancellation cycle is timed, at each place
    of the cycle in turn, and more closely together where the run has fewer
    than 4 pc^2 steps: from pc^2 steps on, every place has its launch."""
    W = pkg.workloads
    mat = W.material(60, seed=5)
    rect, kind, teq, tin = W.ribbon(60.0, 30.0, 6, 300.0, Tinit_first=302.0)
    modes = pkg.ModeTable(ctx, mat["omega"], mat["vx"], mat["vy"], mat["w"], mat["V"], mat["lattz"])
    geom = pkg.Geometry(ctx, rect, kind, teq, tin)
    b = pkg.BertRun(ctx, modes, geom, None, thickness=1.0, dt=4.0, maxtime=4.0 * (steps - 1), max_steps=steps,
                    rta=True, Efactor=4000, Tmax=302.0, Tmin=300.0, seed=3, pcancel_each=pc)
    r = b.execute()
    b.close()
    assert r["nsteps"] == steps and r["step_kernel_timed"] == timed and r["step_kernel_ms"] > 0


@pytest.mark.parametrize("nmodes,threads", [(400, 1024), (4500, 256)])
def test_a_given_capacity_holds_where_velocities_displace_boxes(pkg, ctx, nmodes, threads):
    """4500 modes and 200 boxes do not fit the LDS together. The velocity
    tables alone would, in workgroups whose segments (256 beside 256 of the
    emission) need twice the particles as capacity; those of 256 threads
    (1024 beside 512) need 1.5 times, and a capacity of 1.65 times the
    particles is enough as a tenth of them wait at a wall. 400 modes fit beside
    the boxes, and 2.1 times the particles are given."""
    W = pkg.workloads
    mat = W.material(nmodes, seed=5)
    rect = np.array([[k * 10.0, (k + 1) * 10.0, r * 200.0, r * 200.0 + 100.0] for r in range(4) for k in range(50)])
    modes = pkg.ModeTable(ctx, mat["omega"], mat["vx"], mat["vy"], mat["w"], mat["V"], mat["lattz"])
    geom = pkg.Geometry(ctx, rect, np.zeros(200, np.int32), np.full(200, 300.0), np.full(200, 302.0))

    def run(**kw):
        b = pkg.BertRun(ctx, modes, geom, None, thickness=1.0, dt=4.0, maxtime=8.0, rta=True, Efactor=5000,
                        Tmax=302.0, Tmin=300.0, seed=3, pcancel_each=1000, **kw)
        r = b.execute()
        b.close()
        return r

    a = run()
    n0 = int(a["npart"][0])
    assert n0 > 900000 and a["step_threads"] == 1024
    c = run(capacity=int((2.1 if threads == 1024 else 1.65) * n0))
    assert c["step_threads"] == threads
    assert np.array_equal(a["npart"], c["npart"]) and np.array_equal(a["pending"], c["pending"])
