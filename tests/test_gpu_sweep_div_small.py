"""Compiled sweeps against the oracle bit for bit for numerators down to the smallest subnormal by divisors
above 1 that are no whole numbers: literals, and spacings of uniform meshes."""
import numpy as np
import pytest

import opflow_amd as of
import oracle
from helpers import SEED, build_field
from test_gpu_explicit import DIRC, NEUM, PER, _mesh
from test_gpu_sweep_div import FORMS, _values

pytestmark = pytest.mark.gpu
LITERALS = {
    "literals": lambda u, w: u / 1.35 + w / -1.7 + (u - w) / 7.7 + u / 0.1,
    "literal": lambda u, w: u / 1.35,
    "bounded": lambda u, w: of.conditional(u > w, u / -1.7, of.max(u / 3.3, w)),
}


@pytest.mark.parametrize("mode", [3, 4], ids=["tile", "direct"])
@pytest.mark.parametrize("form", [*LITERALS, "heat", "flux", "weno", "opaque"])
def test_bits_of_the_oracle(ctx, form, mode):
    nodes = [51, 45]
    ctx.set_jit(mode)
    try:
        for ranges in ([(0., 1.35 * 50), (0., 1.7 * 44)], [(-3.3 * 25, 3.3 * 25), (0., 0.3 * 44)]):
            for bc in ([(PER, PER)] * 2, [(DIRC, NEUM), (NEUM, DIRC)]):
                mesh, om = _mesh(ctx, nodes, ranges)
                u, w = (build_field(ctx, mesh, 2, 1, bc, [(0., 0.)] * 2, ext=(3, 3)) for _ in range(2))
                expr = (LITERALS.get(form) or FORMS[form])(u, w)
                flat, flds, root = expr.flatten()
                for n, kind in enumerate(["subnormal", "spread", "tail", "zeros", "ordinary"]):
                    with np.errstate(all="ignore"):
                        a = [oracle.update_padding(f.desc, om, _values(kind, f.shape, SEED + n + 7 * q))
                             for q, f in enumerate((u, w))]
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
