"""The coarse tail of a V-cycle (each cell's stencil in registers): one to three smoothing sweeps on
either side, 2-D and 3-D, coarsest levels of at most 64 cells and of more, every kind of boundary."""
import numpy as np
import pytest

import opflow_amd as of
import oracle

pytestmark = pytest.mark.gpu
D, N_, P = 1, 2, 3
CASES = [([32, 32], [(D, D), (D, D)]), ([64, 32], [(N_, D), (P, P)]), ([52, 36], [(D, N_), (D, D)]),
         ([16, 16, 16], [(D, D), (N_, D), (P, P)]), ([48, 40, 24], [(D, D), (D, N_), (N_, D)]),
         ([20, 12, 36], [(P, P), (D, D), (P, P)])]


@pytest.mark.parametrize("n,bc", CASES, ids=["x".join(map(str, c[0])) for c in CASES])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_sweeps_and_levels(ctx, n, bc, precision):
    """The solution is the oracle's to the bound its own test uses (1e-7 at tolerances 1e-10 and 1e-12),
    and a V-cycle with more sweeps never needs more iterations (one for rounding)."""
    b = np.random.default_rng(11).normal(size=int(np.prod(n)))
    h = [1.0 / n[0]] * len(n)
    ref, _, rel = oracle.pcg_mg(n, h, bc, b, tol=1e-12)
    assert rel <= 1e-12
    g = of.PoissonGMG(ctx, of.poisson_desc(len(n), n, h, bc, 0.0), precision)
    bb, xx = of.DeviceBuffer(ctx, b.size), of.DeviceBuffer(ctx, b.size)
    bb.upload(b)
    its = {}
    for pre, post in ((1, 1), (2, 2), (1, 2), (3, 2), (2, 1), (3, 3)):
        xx.upload(0 * b)
        st = g.solve(bb.ptr, xx.ptr, tol=1e-10, pre=pre, post=post)
        assert st.converged
        assert np.abs(xx.numpy() - ref).max() <= 1e-7 * np.abs(ref).max()
        its[pre, post] = st.niter
    assert its[3, 3] <= its[2, 2] + 1 <= its[1, 1] + 2
    g.close()
    bb.close()
    xx.close()
