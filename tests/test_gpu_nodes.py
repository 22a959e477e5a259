"""updatePadding in one launch: Dirichlet node planes of corner-located dims together with the ghosts
that mirror them, at faces, edges and corners where planes meet, and sizes around a workgroup."""
import itertools

import numpy as np
import pytest

import oracle
from helpers import SEED, build_field, random_storage
from test_gpu_explicit import DIRC, NEUM, PER, _mesh

pytestmark = pytest.mark.gpu
KINDS = [(DIRC, DIRC), (DIRC, NEUM), (NEUM, DIRC), (PER, PER)]


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("nodes", [[6], [257], [5, 7], [33, 9], [260, 6], [6, 5, 7], [9, 14, 6]], ids=str)
def test_planes_and_ghosts(ctx, nodes, dtype):
    mesh, om = _mesh(ctx, nodes, [(0.0, 1.0 + 0.3 * q) for q in range(len(nodes))])
    for n, kinds in enumerate(itertools.product(KINDS, repeat=len(nodes))):
        u = build_field(ctx, mesh, len(nodes), [(n >> q) % 3 == 1 for q in range(len(nodes))] if n % 4 else 0, kinds,
                        [(0.5 + q, -0.25 - q) for q in range(len(nodes))], ext=(2, 2), dtype=dtype)
        raw = random_storage(u, SEED + n).astype(u.dtype)
        u.upload(raw)
        u.updatePadding()
        ref = oracle.update_padding(u.desc, om, raw.astype(np.float64))
        if dtype == "f64":
            np.testing.assert_array_equal(u.numpy(), ref)
        else:  # a rule is three FP32 operations a dim on values of order 1, at most three dims
            np.testing.assert_allclose(u.numpy(), ref, rtol=0, atol=3 * 3 * 4 * 2.0 ** -23 * np.abs(ref).max())
        u.close()
