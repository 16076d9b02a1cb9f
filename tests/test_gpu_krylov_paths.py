"""Routes of the Krylov build around the edges of its kernels."""
import ctypes as C
import threading

import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [0.3, 5.0, 34.0, 40.0])
@pytest.mark.parametrize("m", [2, 3, 15, 16, 17, 30, 32, 33, 63, 64])
def test_small_exponentials(pkg, ctx, m, dt):
    """exp(H) e_1 with 16, 32 or 64 lanes per column, on a number of columns
    that leaves a wave partly empty, with one to 64 applications of the
    Taylor factor and, at dt = 40 ps from the larger m on, by squaring
    (||dt H||_1 above 64). The applications add rounding errors of about
    2^s 20 eps <= 3e-13 relative to a vector of norm <= e^||H|| bounded here
    by the oracle's own; 1e-10 is the tolerance of the other comparisons
    with the oracle's per-column Arnoldi."""
    W = pkg.workloads
    mat, B = W.config1_inputs(nmodes=129, seed=7)
    Po = orc.build_P(B, dt, m, 1)
    Po += (1.0 - Po.sum(0)) / len(B)  # the build's projection to columns summing to 1; the oracle returns V exp(H) e_1
    Pg, rep = pkg.build_P(ctx, B, dt, m=m, precision="fp64", arnoldi="textbook")
    d = np.abs(Pg - Po).max()
    print(f"m={m} dt={dt}: {d:.2e} of {np.abs(Po).max():.2e}", flush=True)
    assert d < 1e-10 * max(1.0, np.abs(Po).max())


def _build(pkg, ctx, B, P, m):
    dp = C.POINTER(C.c_double)
    rep = pkg.KrylovReport()
    pkg.check(pkg.lib().bte_krylov_build(ctx.h, len(B), C.cast(B.ctypes.data, dp), 0.5, m, pkg.PREC["bf16"], 1,
                                         C.cast(P.ctypes.data, dp), C.byref(rep)))


@pytest.mark.parametrize("n", [1447, 1449, 1536])
def test_large_copies(pkg, ctx, n):
    """Operators on both sides of 16 MB, above which pageable memory goes
    through pinned chunks of 4 MB by two threads (N = 1449: the last chunk
    holds 20 kB, N = 1536: half of it is used); pinned memory is copied the
    plain way. The same bits arrive at an output that starts in the middle of a
    page, its neighbours stay as they were, and two threads that share the
    context get the same."""
    hip = C.CDLL("libamdhip64.so.7")  # the one that the library has loaded

    def pinned():
        p = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), C.c_size_t(8 * n * n), 0) == 0
        return p, np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (n, n))

    rng = np.random.default_rng(3)
    B = rng.standard_normal((n, n)) / n
    (hb, pb), (hp, pp) = pinned(), pinned()
    pb[:] = B
    _build(pkg, ctx, pb, pp, 3)
    want = pp.copy()
    assert hip.hipHostFree(hb) == 0 and hip.hipHostFree(hp) == 0
    assert np.isfinite(want).all()
    bufs = [np.full(n * n + 40, 7.0) for _ in range(2)]
    out = [b[17:17 + n * n].reshape(n, n) for b in bufs]
    th = [threading.Thread(target=_build, args=(pkg, ctx, B, o, 3)) for o in out]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for b, o in zip(bufs, out):
        assert np.array_equal(o, want)
        assert (b[:17] == 7.0).all() and (b[17 + n * n:] == 7.0).all()
