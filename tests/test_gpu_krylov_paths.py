"""Routes of the Krylov build around the edges of its kernels."""
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
