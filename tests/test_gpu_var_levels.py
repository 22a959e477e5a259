"""Variable-coefficient 2-D multigrid levels in two launches a level (8 x 8 and 16 x 16 tiles, sides
around and inside a tile, odd coarse sides, every kind of boundary): a known grid function comes back from the
system that the framework's own sweep forms for it."""
import numpy as np
import pytest

import opflow_amd as of
from helpers import SEED

pytestmark = pytest.mark.gpu
D, N, P = of.BCType.Dirc, of.BCType.Neum, of.BCType.Periodic
BCS = {"dirichlet": [(D, D), (D, D)], "mixed": [(D, N), (N, D)], "periodic-x": [(P, P), (D, D)]}


@pytest.mark.parametrize("bc", list(BCS))
@pytest.mark.parametrize("n", [(40, 36), (66, 34), (96, 128), (264, 248), (320, 200), (544, 512)], ids=str)
def test_solution_of_the_discrete_system(ctx, n, bc):
    """div(k grad u) = f with a coefficient of ratio 100. A relative residual of 1e-12 bounds the
    solution's error by 1e-12 times the condition number, about 100 (2 max(n) / pi)^2; twice that for
    the spread of the coefficient over a wavelength."""
    mb = of.MeshBuilder(ctx).newMesh(*[k + 1 for k in n])
    for d in range(2):
        mb.setMeshOfDim(d, 0., n[d] / 128.)
    mesh = mb.build()
    C = of.LocOnMesh.Center

    def field(kinds):
        b = of.ExprBuilder().setMesh(mesh).setLoc([C, C]).setExt(1)
        for d in range(2):
            b.setBC(d, of.DimPos.start, kinds[d][0], 0.).setBC(d, of.DimPos.end, kinds[d][1], 0.)
        return b.build()
    u, f = field(BCS[bc]), field(BCS[bc])
    k = field([(P, P) if BCS[bc][d][0] == P else (N, N) for d in range(2)])
    rng = np.random.default_rng(SEED + n[0])

    def put(x, inner):
        a = np.zeros(x.shape)
        a[1:-1, 1:-1] = inner
        x.upload(a)
        x.updatePadding()
    y, x = np.meshgrid((np.arange(n[1]) + 0.5) / n[1], (np.arange(n[0]) + 0.5) / n[0], indexing="ij")
    put(k, 10.0 ** (np.sin(2 * np.pi * x) * np.cos(2 * np.pi * y)))
    want = np.sin(2 * np.pi * x + 0.3) * np.cos(3 * np.pi * y) + 0.1 * rng.uniform(-1, 1, x.shape)
    put(u, want)
    D1, face = of.D1FirstOrderCentered, of.d1IntpCenterToCorner

    def op(e):
        return of.dx(D1, face(0, k) * of.dx(D1, e)) + of.dy(D1, face(1, k) * of.dy(D1, e))
    f.assign(op(u))
    want = u.numpy()[1:-1, 1:-1]
    put(u, 0.0 * want)
    for precision in ("fp64", "mixed"):
        put(u, 0.0 * want)
        solver = of.makeEqnSolveHandler(lambda e: op(e) == f, u, of.PrecondStructSolver(
            of.StructSolverParams(tol=1e-12, precision=precision)))
        state = solver.solve()
        got = u.numpy()[1:-1, 1:-1]
        assert state.relerr <= 1e-12
        bound = 2 * 1e-12 * 100 * (2 * max(n) / np.pi) ** 2
        assert np.linalg.norm(got - want) <= bound * np.linalg.norm(want)
