"""The sweep interpreter's bundled form against the oracle, bit for bit: numbers of loads around its
groups (1, 4, 8, 16), more values than it holds (the stack program), cells around a wave and rows that
end inside one, several waves a workgroup."""
import numpy as np
import pytest

import opflow_amd as of
from helpers import SEED
from test_gpu_explicit import PER, _sweep_case

pytestmark = pytest.mark.gpu
SPEC = (1, [(PER, PER)] * 3, None, (4, 4))


@pytest.fixture(autouse=True)
def interpreter(ctx):
    ctx.set_jit(0)
    yield
    ctx.set_jit(1)


@pytest.mark.parametrize("fields", [1, 2])
@pytest.mark.parametrize("window", [(1, 1), (3, 1), (1, 5), (7, 1), (3, 3), (9, 1), (3, 5), (5, 5), (9, 3), (7, 7),
                                    (9, 9)], ids=str)
def test_numbers_of_loads(ctx, window, fields):
    w = np.random.default_rng(SEED).uniform(-1, 1, window)

    def fn(u, v=None):
        return of.conv(u, w) if v is None else of.conv(u, w) - of.conv(v, w) / 3.0
    got, ref = _sweep_case(ctx, fn, [SPEC] * fields, [14, 12], SPEC, SEED + sum(window))
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("nodes", [[9, 9], [14, 6], [65, 6], [66, 9], [8, 129], [301, 250], [513, 521], [30, 21, 12]], ids=str)
def test_sizes(ctx, nodes):
    D2, W, UP = of.D2SecondOrderCentered, of.D1WENO53Upwind, of.D1FirstOrderBiasedUpwind

    def fn(u, w):
        e = u + 0.01 * (of.d2x(D2, u) + of.d2y(D2, w)) - 0.1 * of.dx(W, u) * of.dy(UP, w)
        return of.conditional(u > w, e, e / 3.0 - of.abs(of.min(u, w)))
    got, ref = _sweep_case(ctx, fn, [SPEC, SPEC], nodes, None, SEED + 2)
    np.testing.assert_array_equal(got, ref)
