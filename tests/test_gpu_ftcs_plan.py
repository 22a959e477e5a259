"""Steps a launch of the 2-D heat kernel takes on grids past the caches, where a launch costs a pass over
memory: the plan has to count it."""
import pytest

import opflow_amd as of
from helpers import build_field
from test_gpu_explicit import PER, _mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n,span,least", [(4096, 1.0, 6), (8192, 1.0, 6), (8000, 1.0, 4), (3000, 1.0, 4)], ids=str)
def test_large_grids_take_several_steps(ctx, n, span, least, dtype):
    """A step of a launch of nt steps moves about 2 / nt fields. With the fields past the L2s that is
    the larger part of a step below 4 (divisions by a spacing that is no power of two) or 6."""
    mesh, _ = _mesh(ctx, [n + 1, n + 1], [(0., span)] * 2)
    u = build_field(ctx, mesh, 2, 1, [(PER, PER)] * 2, None, dtype=dtype)
    launches, most = u.ftcs_plan(240)
    u.close()
    assert least <= most <= 24 and launches == -(-240 // most)
