"""2-D FTCS steps in registers: sides around the 64- and 128-cell regions and their wave rows, every
kind of side, step counts of one and of several launches; values outside the range in which the
divisions by a spacing go through its reciprocal."""
import numpy as np
import pytest

import opflow_amd as of
import oracle
from helpers import build_field, SEED
from test_gpu_explicit import _mesh

pytestmark = pytest.mark.gpu
DIRC, NEUM, PER = 1, 2, 3

SIDES = [(5, 5), (6, 7), (7, 30), (5, 29), (61, 28), (62, 29), (63, 61), (64, 62), (65, 31), (62, 300), (300, 29),
         (127, 63), (131, 97), (190, 258)]
BCS = [[(DIRC, DIRC), (DIRC, DIRC)], [(PER, PER), (DIRC, NEUM)], [(NEUM, DIRC), (PER, PER)], [(PER, PER), (PER, PER)]]


def _run(ctx, n, ranges, bc, bcv, init, coef, steps, tblock=0, dtype="f64"):
    mesh, om = _mesh(ctx, [m + 1 for m in n], ranges)
    u = build_field(ctx, mesh, 2, 1, bc, bcv, dtype=dtype)
    init = oracle.update_padding(u.desc, om, np.asarray(init(u), dtype=np.float64))
    u.upload(init)
    u.ftcs_blocked(coef, steps, tblock)
    got = u.numpy()
    u.close()
    return got, init, u.desc, om


@pytest.mark.parametrize("bc", range(len(BCS)))
@pytest.mark.parametrize("n", SIDES, ids=[f"{a}x{b}" for a, b in SIDES])
def test_bits_of_the_oracle(ctx, n, bc):
    for ranges, steps, tblock in (([(0., 1.3), (0., 0.7)], 13, 0), ([(0., n[0] / 64.), (0., n[1] / 64.)], 21, 0),
                                  ([(0., n[0] / 64.), (0., n[1] / 32.)], 2, 0), ([(0.1, 1.3), (0., 1.)], 150, 0),
                                  ([(0., 1.), (0., 1.)], 2, 1)):
        h = [(r[1] - r[0]) / m for r, m in zip(ranges, n)]
        coef = 0.4 / sum(1 / a ** 2 for a in h)
        rng = np.random.default_rng(SEED + n[0])
        got, init, d, om = _run(ctx, n, ranges, BCS[bc], [(0.3, -0.5), (0.25, 0.)],
                                lambda u: rng.uniform(-1, 1, u.shape), coef, steps, tblock)
        np.testing.assert_array_equal(got, oracle.ftcs(d, om, init, coef, steps))


@pytest.mark.parametrize("n", [(500, 460), (1030, 1100), (2100, 2050)], ids=str)
def test_larger_regions(ctx, n):
    for ranges in ([(0., 1.), (0., 1.)], [(0., n[0] / 512.), (0., n[1] / 512.)]):
        h = [(r[1] - r[0]) / m for r, m in zip(ranges, n)]
        coef = 0.4 / sum(1 / a ** 2 for a in h)
        rng = np.random.default_rng(SEED)
        got, init, d, om = _run(ctx, n, ranges, BCS[0], [(0.3, -0.5), (0.25, 0.)],
                                lambda u: rng.uniform(-1, 1, u.shape), coef, 25)
        np.testing.assert_array_equal(got, oracle.ftcs(d, om, init, coef, 25))


def _float_reference(init, n, h, per, bcv, coef, steps):
    """The reference's operations in float32 (spacings and coefficient rounded to float)."""
    f = np.float32
    u, hx, hy, coef = init.astype(f), f(h[0]), f(h[1]), f(coef)

    def fill(a, q, d):
        lo, hi = [slice(None)] * 2, [slice(None)] * 2
        at = lambda i: tuple(i if k == q else slice(None) for k in range(2))  # noqa: E731
        if per[d]:
            a[at(0)], a[at(-1)] = a[at(-2)].copy(), a[at(1)].copy()
    for _ in range(steps):
        c = u[1:-1, 1:-1]
        dx = ((u[1:-1, 2:] - c) / hx - (c - u[1:-1, :-2]) / hx) / hx
        dy = ((u[2:, 1:-1] - c) / hy - (c - u[:-2, 1:-1]) / hy) / hy
        u = u.copy()
        u[1:-1, 1:-1] = c + coef * (dx + dy)
        fill(u, 1, 0)
        fill(u, 0, 1)
    return u


@pytest.mark.parametrize("scale", [1.0, 1e-30, 3e-37, 1e-42, 1e30])
def test_float_bits(ctx, scale):
    """FP32 against the same operations in numpy, down to subnormal quotients."""
    n = (150, 70)
    h = [1. / m for m in n]
    coef = 0.4 / sum(1 / a ** 2 for a in h)
    rng = np.random.default_rng(SEED)
    got, init, d, om = _run(ctx, n, None, BCS[3], None,
                            lambda u: (rng.uniform(-1, 1, u.shape) * scale).astype(np.float32), coef, 9, dtype="f32")
    with np.errstate(all="ignore"):
        ref = _float_reference(init, n, h, (True, True), None, coef, 9)
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("case", ["tiny", "spread", "subnormal", "huge", "gap", "special", "decay"])
def test_values_outside_the_range(ctx, case):
    n = (190, 75)
    rng = np.random.default_rng(SEED + 5)

    def init(u):
        v = rng.uniform(-1, 1, u.shape)
        if case == "tiny":
            return v * 1e-301
        if case == "spread":
            return v * 10.0 ** rng.integers(-320, 10, u.shape).astype(float)
        if case == "subnormal":
            return rng.integers(-5000, 5000, u.shape) * 5e-324
        if case == "huge":
            return v * 1e307
        if case == "gap":  # zeros beside ordinary values: the pulse's front decays step by step
            return np.where(np.abs(np.arange(u.shape[1]) - 90)[None, :] + 0 * v < 3, v, 0.0)
        if case == "decay":
            return np.exp(-((np.arange(u.shape[1]) - 90.0) ** 2)[None, :] / 12.0) * (1 + 0 * v)
        w = v.copy()
        w[20:23, 30:33], w[50, 100], w[60, 10] = np.inf, np.nan, -0.0
        return w
    coef = 0.4 / sum(m ** 2 for m in n)
    with np.errstate(all="ignore"):
        for bc, bcv in ((BCS[0], [(0., 0.), (1e-200, 1e-320)]), (BCS[3], None)):
            got, start, d, om = _run(ctx, n, None, bc, bcv, init, coef, 60)
            np.testing.assert_array_equal(got, oracle.ftcs(d, om, start, coef, 60))
