"""FP32 heat steps with Dirichlet constants and Neumann slopes down to the smallest subnormal, on spacings
whose quotients then fall midway between two floats, against the same operations in numpy."""
import numpy as np
import pytest

from helpers import build_field, SEED
from test_gpu_explicit import _mesh

pytestmark = pytest.mark.gpu
DIRC, NEUM, PER = 1, 2, 3
F = np.float32


def _fill(u, h, bc, bcv):
    """updatePadding's rules in float32 (axis 0 of the storage is the last dimension)."""
    dim = u.ndim
    for d in range(dim):
        def at(i):
            return tuple(i if q == dim - 1 - d else slice(None) for q in range(dim))
        if bc[d][0] == PER:
            u[at(0)], u[at(-1)] = u[at(-2)].copy(), u[at(1)].copy()
            continue
        for s, (ghost, cell, sign) in enumerate(((0, 1, 1.0), (-1, -2, -1.0))):
            g = bcv[d][s]
            if bc[d][s] == DIRC:  # the line through the wall's value and the cell's
                a, b = sign * h[d] / 2, sign * h[d]
                u[at(ghost)] = (F(a) * u[at(cell)] - F(b * g)) / F(a - b)
            else:
                u[at(ghost)] = u[at(cell)] + F(-sign * h[d] * g)
    return u


def _step(u, h, coef):
    dim = u.ndim
    inner = tuple(slice(1, -1) for _ in range(dim))
    c, acc = u[inner], None
    for d in range(dim):
        def at(lo, hi):
            return tuple(slice(lo, hi) if q == dim - 1 - d else slice(1, -1) for q in range(dim))
        q = ((u[at(2, None)] - c) / F(h[d]) - (c - u[at(0, -2)]) / F(h[d])) / F(h[d])
        acc = q if acc is None else acc + q
    u = u.copy()
    u[inner] = c + F(coef) * acc
    return u


CASES = [((70, 41), [(DIRC, DIRC), (DIRC, NEUM)]), ((5, 7), [(DIRC, NEUM), (DIRC, DIRC)]),
         ((9, 6, 11), [(DIRC, DIRC)] * 3), ((66, 5, 7), [(PER, PER), (DIRC, DIRC), (NEUM, DIRC)])]


@pytest.mark.parametrize("h", [(196., 392., 300.), (300., 196., 308.), (3., 7., 24.)], ids=str)
@pytest.mark.parametrize("case", range(len(CASES)))
def test_float_bits(ctx, case, h):
    n, bc = CASES[case]
    dim = len(n)
    h = list(h[:dim])
    unit = 2.0 ** -149
    rng = np.random.default_rng(SEED + case)
    mesh, _ = _mesh(ctx, [m + 1 for m in n], [(0., a * m) for a, m in zip(h, n)])
    coef = 0.4 / sum(1 / a ** 2 for a in h)
    for k in range(12):
        scale = 2.0 ** (2 * k)  # from a unit's quarter to the normal numbers
        bcv = [[0.25 * unit * scale * int(rng.integers(1, 400)) for _ in range(2)] for _ in range(dim)]
        u = build_field(ctx, mesh, dim, 1, bc, bcv, dtype="f32")
        start = np.where(rng.random(u.shape) < 0.8, 0.0, rng.uniform(-1, 1, u.shape) * (k & 1)).astype(F)
        with np.errstate(all="ignore"):
            ref = _fill(start.copy(), h, bc, bcv)
            u.upload(ref.astype(u.dtype))
            u.updatePadding()
            np.testing.assert_array_equal(u.numpy(), ref)  # the rules themselves, by the ghost launch
            u.ftcs_blocked(coef, 5, 0)
            for _ in range(5):
                ref = _fill(_step(ref, h, coef), h, bc, bcv)
        np.testing.assert_array_equal(u.numpy(), ref, err_msg=f"k {k} {bcv}")
        u.close()
