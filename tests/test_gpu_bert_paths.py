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
