"""3-D FTCS steps in registers: sides around the 64 x 64 region and its waves' four rows, few and many
planes, every kind of side, step counts of one and of several launches; values outside the range in
which the divisions by a spacing go through its reciprocal."""
import numpy as np
import pytest

import opflow_amd as of
import oracle
from helpers import build_field, SEED
from test_gpu_explicit import _mesh
from test_gpu_ftcs2d import DIRC, NEUM, PER

pytestmark = pytest.mark.gpu

SIDES = [(5, 5, 5), (7, 57, 6), (58, 5, 9), (59, 60, 5), (61, 62, 7), (62, 63, 11), (64, 65, 5), (117, 59, 13),
         (130, 121, 6)]
BCS = [[(DIRC, DIRC)] * 3, [(PER, PER), (DIRC, NEUM), (NEUM, DIRC)], [(NEUM, DIRC), (PER, PER), (DIRC, DIRC)],
       [(DIRC, NEUM), (DIRC, DIRC), (PER, PER)], [(PER, PER)] * 3]
VALUES = [(0.3, -0.5), (0.25, 0.), (-0.75, 1.5)]


def _run(ctx, n, h, bc, bcv, init, coef, steps, tblock=0, dtype="f64"):
    mesh, om = _mesh(ctx, [m + 1 for m in n], [(0., a * m) for a, m in zip(h, n)])
    u = build_field(ctx, mesh, 3, 1, bc, bcv, dtype=dtype)
    init = np.asarray(init(u), dtype=np.float64)
    init = oracle.update_padding(u.desc, om, init)
    u.upload(init)
    u.ftcs_blocked(coef, steps, tblock)
    got = u.numpy()
    u.close()
    return got, init, u.desc, om


@pytest.mark.parametrize("bc", range(len(BCS)))
@pytest.mark.parametrize("n", SIDES, ids=str)
def test_bits_of_the_oracle(ctx, n, bc):
    for h, steps, tblock in (((0.013, 0.007, 0.021), 7, 0), ((1 / 64.,) * 3, 4, 0), ((1 / 64., 1 / 32., 1 / 64.), 2, 0),
                             ((0.1, 0.3, 0.2), 1, 0), ((0.1, 0.1, 0.1), 3, 1)):
        coef = 0.4 / sum(1 / a ** 2 for a in h)
        rng = np.random.default_rng(SEED + n[0])
        got, init, d, om = _run(ctx, n, h, BCS[bc], VALUES, lambda u: rng.uniform(-1, 1, u.shape), coef, steps, tblock)
        np.testing.assert_array_equal(got, oracle.ftcs(d, om, init, coef, steps))


def _float_reference(init, h, coef, steps):
    """The reference's operations in float32, every dimension periodic."""
    f = np.float32
    u, hx, hy, hz, coef = init.astype(f), f(h[0]), f(h[1]), f(h[2]), f(coef)
    for _ in range(steps):
        c = u[1:-1, 1:-1, 1:-1]
        dx = ((u[1:-1, 1:-1, 2:] - c) / hx - (c - u[1:-1, 1:-1, :-2]) / hx) / hx
        dy = ((u[1:-1, 2:, 1:-1] - c) / hy - (c - u[1:-1, :-2, 1:-1]) / hy) / hy
        dz = ((u[2:, 1:-1, 1:-1] - c) / hz - (c - u[:-2, 1:-1, 1:-1]) / hz) / hz
        u = np.pad(c + coef * ((dx + dy) + dz), 1, mode="wrap")
    return u


@pytest.mark.parametrize("scale", [1.0, 1e-30, 3e-37, 1e-42, 1e30])
@pytest.mark.parametrize("h", [(0.013, 0.007, 0.021), (7., 9., 11.), (3e4, 1e-3, 1.)], ids=str)
def test_float_bits(ctx, h, scale):
    """FP32 against the same operations in numpy, down to subnormal quotients."""
    n = (70, 66, 9)
    coef = 0.4 / sum(1 / a ** 2 for a in h)
    rng = np.random.default_rng(SEED)
    got, init, d, om = _run(ctx, n, h, BCS[4], None,
                            lambda u: (rng.uniform(-1, 1, u.shape) * scale).astype(np.float32), coef, 7, dtype="f32")
    with np.errstate(all="ignore"):
        np.testing.assert_array_equal(got, _float_reference(init, [a * m / m for a, m in zip(h, n)], coef, 7))


@pytest.mark.parametrize("case", ["tiny", "subnormal", "huge", "gap", "special"])
def test_values_outside_the_range(ctx, case):
    n = (66, 61, 12)
    rng = np.random.default_rng(SEED + 5)

    def init(u):
        v = rng.uniform(-1, 1, u.shape)
        if case == "tiny":
            return v * 1e-301
        if case == "subnormal":
            return rng.integers(-5000, 5000, u.shape) * 5e-324
        if case == "huge":
            return v * 1e307
        if case == "gap":  # zeros beside ordinary values: the front decays step by step
            return np.where(np.abs(np.arange(u.shape[2]) - 30)[None, None, :] + 0 * v < 3, v, 0.0)
        w = v.copy()
        w[5, 20:23, 30:33], w[3, 50, 60], w[7, 60, 10] = np.inf, np.nan, -0.0
        return w
    h = (0.013, 0.007, 0.021)
    coef = 0.4 / sum(1 / a ** 2 for a in h)
    with np.errstate(all="ignore"):
        for bc, bcv in ((BCS[0], [(0., 0.), (1e-200, 1e-320), (0., 0.)]), (BCS[4], None)):
            got, start, d, om = _run(ctx, n, h, bc, bcv, init, coef, 25)
            np.testing.assert_array_equal(got, oracle.ftcs(d, om, start, coef, 25))
