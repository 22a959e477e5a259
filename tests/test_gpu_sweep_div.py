"""Compiled sweeps against the oracle bit for bit where divisions go through a reciprocal or a known
spacing: uniform spacings that are no power of two, literals, WENO's weights, coordinates that are whole
multiples of a power-of-two spacing or not; values outside the range the reciprocals are good for."""
import numpy as np
import pytest

import opflow_amd as of
import oracle
from helpers import SEED, build_field
from test_gpu_explicit import DIRC, NEUM, PER, _mesh

pytestmark = pytest.mark.gpu
D1, D2, W, V = of.D1FirstOrderCentered, of.D2SecondOrderCentered, of.D1WENO53Upwind, of.D1WENO53Downwind
C2N, N2C = of.d1IntpCenterToCorner, of.d1IntpCornerToCenter
FORMS = {
    "heat": lambda u, w: u + 1e-4 * (of.d2x(D2, u) + of.d2y(D2, u)),
    "flux": lambda u, w: u + 1e-4 * (of.dx(D1, C2N(0, w) * of.dx(D1, u)) + of.dy(D1, C2N(1, w) * of.dy(D1, u))),
    "weno": lambda u, w: u - 1e-3 * (of.dx(W, u) + w * of.dy(V, u)),
    "literal": lambda u, w: u / 3.0 - w / -7.0 + (u - w) / 0.1 + u / 1e200 + w / 0.25,
    "opaque": lambda u, w: of.conditional(u > of.dx(of.D1FirstOrderBiasedUpwind, w), u / 3.0, of.max(of.d2y(D2, u), w)),
}
RANGES = [[(0., 1.), (0., 1.)], [(0., 0.25), (-0.5, 0.5)], [(0.3, 1.3), (0.1, 0.35)]]
VALUES = ["ordinary", "zeros", "tiny", "subnormal", "huge", "special", "spread", "tail"]


def _values(kind, shape, seed):
    rng = np.random.default_rng(seed)
    v = rng.uniform(-1, 1, shape)
    if kind == "zeros":
        return np.where(rng.random(shape) < 0.7, 0.0, v) * np.where(rng.random(shape) < 0.5, -1.0, 1.0)
    if kind == "subnormal":
        return rng.integers(-9000, 9000, shape) * 5e-324
    if kind == "special":
        v[tuple(n // 2 for n in shape)], v[tuple(n // 3 for n in shape)] = np.inf, np.nan
        return v
    if kind == "spread":
        return v * 10.0 ** rng.integers(-320, 300, shape).astype(float)
    if kind == "tail":
        return np.exp(-40.0 * np.arange(v.size).reshape(shape) / shape[-1]) * 1e-60
    return v * {"ordinary": 1.0, "tiny": 1e-250, "huge": 1e290}[kind]


@pytest.mark.parametrize("mode", [3, 4], ids=["tile", "direct"])
@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("nodes", [[65, 33], [51, 45]], ids=str)
def test_bits_of_the_oracle(ctx, nodes, form, mode):
    ctx.set_jit(mode)
    try:
        for ranges in RANGES:
            for bc in ([(PER, PER)] * 2, [(DIRC, NEUM), (NEUM, DIRC)]):
                mesh, om = _mesh(ctx, nodes, ranges)
                u, w = (build_field(ctx, mesh, 2, 1, bc, [(0., 0.)] * 2, ext=(3, 3)) for _ in range(2))
                expr = FORMS[form](u, w)
                flat, flds, root = expr.flatten()
                for n, kind in enumerate(VALUES):
                    with np.errstate(all="ignore"):
                        a = [oracle.update_padding(f.desc, om, _values(k, f.shape, SEED + n))
                             for f, k in ((u, kind), (w, "ordinary" if n % 2 else kind))]
                        u.upload(a[0])
                        w.upload(a[1])
                        arrays = {id(u): a[0], id(w): a[1]}
                        ref = oracle.assign(flat, root, [(arrays[id(f)], f.desc) for f in flds], om, a[0], u.desc, 0,
                                            update_padding=lambda r: oracle.update_padding(u.desc, om, r))
                    u.assign(expr)
                    np.testing.assert_array_equal(u.numpy(), ref, err_msg=f"{kind} {ranges}")
                u.close()
                w.close()
    finally:
        ctx.set_jit(1)


def test_tiles_in_3d(ctx):
    ctx.set_jit(3)
    try:
        for nodes, ranges in (([33, 17, 9], [(0., 1.), (0., 0.5), (-1., 1.)]), ([30, 21, 12], None)):
            mesh, om = _mesh(ctx, nodes, ranges)
            u, w = (build_field(ctx, mesh, 3, 1, [(PER, PER)] * 3, None, ext=(3, 3)) for _ in range(2))
            expr = u + 1e-4 * sum((of.d1(D1, d, C2N(d, w) * of.d1(D1, d, u)) for d in range(3)), 0.0) - 1e-3 * of.dz(W, u)
            flat, flds, root = expr.flatten()
            a = [oracle.update_padding(f.desc, om, _values("ordinary", f.shape, SEED + k)) for k, f in enumerate((u, w))]
            u.upload(a[0])
            w.upload(a[1])
            arrays = {id(u): a[0], id(w): a[1]}
            ref = oracle.assign(flat, root, [(arrays[id(f)], f.desc) for f in flds], om, a[0], u.desc, 0,
                                update_padding=lambda r: oracle.update_padding(u.desc, om, r))
            u.assign(expr)
            np.testing.assert_array_equal(u.numpy(), ref)
            u.close()
            w.close()
    finally:
        ctx.set_jit(1)
