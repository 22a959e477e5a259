"""3-D V(2,2) levels in two launches (cubes of 8 x 8 x 8 cells and remainders of them) with a shift and
every kind of side: solutions against the cell-by-cell operator of the oracle."""
import numpy as np
import pytest

import opflow_amd as of
import oracle

pytestmark = pytest.mark.gpu
D, N, P = 1, 2, 3


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("sigma", [0.0, 0.75])
@pytest.mark.parametrize("n", [(20, 24, 28), (36, 40, 44), (64, 48, 32), (72, 80, 56), (96, 64, 64)], ids=str)
@pytest.mark.parametrize("bc", [[(D, D)] * 3, [(D, N), (P, P), (N, N)], [(P, P), (D, D), (N, D)]],
                         ids=["dirichlet", "mixed", "periodic-x"])
def test_residual_of_the_operator(ctx, n, bc, sigma, precision):
    h = [1.0 / k for k in n]
    b = np.random.default_rng(sum(n)).standard_normal(n[::-1])
    g = of.PoissonGMG(ctx, of.poisson_desc(3, list(n), h, bc, sigma), precision)
    bb, xx = of.DeviceBuffer(ctx, b.size), of.DeviceBuffer(ctx, b.size)
    bb.upload(b.ravel())
    xx.upload(np.zeros(b.size))
    st = g.solve(bb.ptr, xx.ptr, tol=1e-9, max_iter=60)
    x = xx.numpy()
    r = b.ravel() - oracle.poisson_apply(list(n), h, bc, x.ravel(), sigma)
    # the solve's own test with the rounding of A x: ||A|| ||x|| <= 4 sum(1 / h^2) ||x||
    slack = 16 * 2.0 ** -53 * 4 * sum(k * k for k in n) * np.linalg.norm(x)
    assert st.converged and np.linalg.norm(r) <= 1e-9 * np.linalg.norm(b) + slack
    # a V(2,2) cycle halves the residual at least, at spacings of up to 1 : 2 (nine digits: 30 cycles)
    assert st.niter <= 30
    g.close(), bb.close(), xx.close()
