"""The splat over points sorted by brick and cell (gfsx_splat.hip) against
the oracle: ragged grids, empty, crowded and overfull bricks, radii of one to
several nodes, points outside the bins."""
import numpy as np
import pytest

from conftest import NORM_REL_TOL, norm_rel

pytestmark = pytest.mark.gpu


def points(dims, dx, n, crowd, seed):
    rng = np.random.default_rng(seed)
    ext = np.array(dims) * dx
    pos = rng.uniform(-0.1, 1.1, size=(n, 3)) * ext
    # one cell with most of the crowd, and the brick around it
    c = np.array(dims) // 2
    pos[:crowd] = (c + rng.uniform(0.02, 0.98, size=(crowd, 3))) * dx
    pos[: crowd // 4] = (c + rng.uniform(-2.0, 3.0, size=(crowd // 4, 3))) * dx
    if n > 20:
        pos[-20:-10] = np.round(pos[-20:-10] / dx) * dx
    pos = pos[rng.permutation(n)].astype(np.float32)
    return pos, rng.normal(size=n).astype(np.float32)


@pytest.mark.parametrize("dims,n,crowd,radius", [
    ((1, 1, 1), 1, 0, 1.0),
    ((7, 8, 9), 500, 0, 1.0),
    ((17, 9, 24), 9000, 1200, 1.7),
    ((25, 33, 16), 30000, 9000, 1.0),    # a brick past the LDS capacity
    ((20, 21, 22), 8000, 700, 3.0),
    ((130, 16, 70), 20011, 0, 2.5),
])
def test_splat_matches_oracle(ctx, orc, dims, n, crowd, radius):
    dx, off = 0.1, (0.0, 0.05, -0.03)
    pos, val = points(dims, dx, n, crowd, 21)
    S, W = ctx.p2g(pos, val, radius * dx, off, dx, dims)
    Se, We = orc.p2g(pos, val, radius * dx, off, dx, dims)
    assert norm_rel(S, Se) <= NORM_REL_TOL and norm_rel(W, We) <= NORM_REL_TOL
    S2, W2 = ctx.p2g(pos, val, radius * dx, off, dx, dims)
    assert np.array_equal(S, S2) and np.array_equal(W, W2)
    P, _ = ctx.p2g(pos, None, radius * dx, off, dx, dims, weight=False)
    assert norm_rel(P, We) <= NORM_REL_TOL     # the weight alone
