"""The coarsest level's dense inverse, through solves whose hierarchy is that one level (an odd
side cannot be coarsened): sizes around the 32-cell pivot blocks and 64-cell tiles up to the 1024
cells the solver takes, singular operators and an indefinite one."""
import numpy as np
import pytest

import opflow_amd as of
import oracle

pytestmark = pytest.mark.gpu
D, N_, P = 1, 2, 3

CASES = [([5, 3], [(D, D)] * 2, 0.0), ([8, 8], [(D, N_), (D, D)], 0.0), ([9, 7], [(D, D), (P, P)], 0.0),
         ([5, 13], [(D, D)] * 2, 3.0), ([25, 40], [(N_, D), (D, D)], 0.0), ([31, 33], [(D, D)] * 2, 0.0),
         ([7, 9, 16], [(D, D), (N_, N_), (P, P)], 0.0), ([31, 33], [(N_, N_)] * 2, 0.0),
         ([9, 11, 7], [(P, P)] * 3, 0.0), ([21, 17], [(D, D)] * 2, -60.0)]


@pytest.mark.parametrize("n,bc,sigma", CASES, ids=[f"{'x'.join(map(str, c[0]))}-{i}" for i, c in enumerate(CASES)])
def test_one_level_solve_is_the_dense_solve(ctx, n, bc, sigma):
    N = int(np.prod(n))
    h = [1.0 / n[0]] * len(n)
    A = np.stack([oracle.poisson_apply(n, h, bc, e, sigma=sigma) for e in np.eye(N)], axis=1)
    w, V = np.linalg.eigh(A)
    singular = np.abs(w) < 1e-9 * np.abs(w).max()
    assert (singular.sum() == 1) == (sigma == 0.0 and all(t in (N_, P) for p in bc for t in p))
    assert (w.min() < -1e-9 * w.max()) == (sigma < 0)
    b = np.random.default_rng(3).normal(size=N)
    if singular.any():
        b -= b.mean()
    tol = 1e-12
    g = of.PoissonGMG(ctx, of.poisson_desc(len(n), n, h, bc, sigma), "fp64")
    bb, xx = of.DeviceBuffer(ctx, N), of.DeviceBuffer(ctx, N)
    bb.upload(b)
    st = g.solve(bb.ptr, xx.ptr, tol=tol)
    x = xx.numpy()
    g.close(); bb.close(); xx.close()
    assert st.converged and st.niter <= 3  # the preconditioner is the inverse
    c = np.where(singular, 0.0, V.T @ b / np.where(singular, 1.0, w))
    ref = V @ c
    if singular.any():
        x = x - x.mean()
    # |x - ref| <= |A^-1| |residual|, the residual within tol |b|; twice that for the rounding of ref
    assert np.linalg.norm(x - ref) <= 2 * tol * np.linalg.norm(b) / np.abs(w[~singular]).min()
