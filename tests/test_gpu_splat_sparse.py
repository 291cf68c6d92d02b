"""The splat's two gathers (by rows, or a plane's rows as one sequence where no
brick holds more than 1024 points) at their line, over the radii' cell spans,
clipped and brick-crossing rows, against the oracle."""
import numpy as np
import pytest

from conftest import NORM_REL_TOL, norm_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("radius", [1.0, 1.6, 2.5, 3.5, 4.0])
@pytest.mark.parametrize("crowd", [0, 1, 1023, 1024, 1025])
def test_splat_sparse_line(ctx, orc, radius, crowd):
    dims, dx, off = (37, 20, 21), 0.125, (0.0, 0.0, 0.0)
    rng = np.random.default_rng(crowd)
    # the crowd in one 8-cell brick of the bins whatever their pad (0..4)
    near = rng.uniform(8.02, 11.98, size=(crowd, 3))
    far = np.concatenate([rng.uniform(16.02, 36.9, size=(700, 1)),
                          rng.uniform(-1.0, 21.0, size=(700, 2))], axis=1)
    pos = (rng.permutation(np.concatenate([near, far])) * dx).astype(np.float32)
    val = rng.normal(size=len(pos)).astype(np.float32)
    S, W = ctx.p2g(pos, val, radius * dx, off, dx, dims)
    Se, We = orc.p2g(pos, val, radius * dx, off, dx, dims)
    assert norm_rel(S, Se) <= NORM_REL_TOL and norm_rel(W, We) <= NORM_REL_TOL
    P, _ = ctx.p2g(pos, None, radius * dx, off, dx, dims, weight=False)
    assert norm_rel(P, We) <= NORM_REL_TOL
