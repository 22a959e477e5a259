"""The interpreter's two forms in FP32 around the line between them (cells a compute unit, bundles against
instructions): the bits of the same operations in numpy, and of the compiled sweep."""
import numpy as np
import pytest

import opflow_amd as of
from helpers import SEED, build_field
from test_gpu_explicit import PER, _mesh

pytestmark = pytest.mark.gpu
D1, D2 = of.D1FirstOrderCentered, of.D2SecondOrderCentered


def _horner(k):
    def fn(u, w):
        e = u
        for q in range(k):
            e = e * w + (1.5 + q)
        return e
    return fn


def _numpy_horner(k, u, w):
    e = u
    for q in range(k):
        e = e * w + np.float32(1.5 + q)
    return e


STENCILS = {
    "dx": lambda u, w: of.dx(D1, u),
    "two": lambda u, w: u - 0.1 * (w * of.dx(D1, u) + w * of.dy(D1, u)),
    "d2x": lambda u, w: of.d2x(D2, u),
    "heat": lambda u, w: u + 0.01 * (of.d2x(D2, u) + of.d2y(D2, u)),
    "select": lambda u, w: of.conditional(u > w, of.max(u, 0.5 * w), of.abs(u) / 3.0),
}


# 24 waves a compute unit of 256 are 393216 cells: one row below and above, and far on both sides
@pytest.mark.parametrize("n", [(70, 33), (640, 614), (640, 615), (1001, 777), (64, 64, 97)], ids=str)
def test_bits(ctx, n):
    mesh, _ = _mesh(ctx, [m + 1 for m in n])
    dim = len(n)
    u, w, a, b = (build_field(ctx, mesh, dim, 1, [(PER, PER)] * dim, None, dtype="f32") for _ in range(4))
    rng = np.random.default_rng(SEED + n[0])
    for f in (u, w):
        f.upload(rng.uniform(-1, 1, f.shape).astype(np.float32))
        f.updatePadding()
    inner = (slice(1, -1),) * dim
    try:
        for k in (1, 2, 7, 20):
            ctx.set_jit(0)
            a.assign(_horner(k)(u, w))
            np.testing.assert_array_equal(a.numpy()[inner], _numpy_horner(k, u.numpy()[inner], w.numpy()[inner]))
        for name, fn in STENCILS.items():
            ctx.set_jit(0)
            a.assign(fn(u, w))
            ctx.set_jit(4)
            b.assign(fn(u, w))
            np.testing.assert_array_equal(a.numpy(), b.numpy(), err_msg=name)
    finally:
        ctx.set_jit(1)
        for f in (u, w, a, b):
            f.close()
