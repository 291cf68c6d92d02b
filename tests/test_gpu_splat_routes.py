"""The splat on both sides of the lines between its two sorts, against the
oracle: brick histograms in LDS for radii of up to 4 cells and fewer than 40000
bricks of 8^3 bin cells, the cell sort and its gather beyond."""
import numpy as np
import pytest

from conftest import NORM_REL_TOL, norm_rel

pytestmark = pytest.mark.gpu


def check(ctx, orc, dims, n, radius, seed):
    dx, off = 0.1, (0.0, 0.05, -0.03)
    rng = np.random.default_rng(seed)
    pos = (rng.uniform(-0.05, 1.05, size=(n, 3)) * np.array(dims) * dx).astype(np.float32)
    val = rng.normal(size=n).astype(np.float32)
    S, W = ctx.p2g(pos, val, radius * dx, off, dx, dims)
    Se, We = orc.p2g(pos, val, radius * dx, off, dx, dims)
    assert norm_rel(S, Se) <= NORM_REL_TOL and norm_rel(W, We) <= NORM_REL_TOL
    P, _ = ctx.p2g(pos, None, radius * dx, off, dx, dims, weight=False)
    assert norm_rel(P, We) <= NORM_REL_TOL


@pytest.mark.parametrize("radius", [3.99, 4.01, 4.3, 6.0])
@pytest.mark.parametrize("dims,n", [((23, 18, 20), 3000), ((9, 40, 11), 500), ((1, 1, 1), 3)])
def test_radius_line(ctx, orc, dims, n, radius):
    check(ctx, orc, dims, n, radius, 3)


# R = dx adds one bin cell an axis: 31*24*22 = 16368 bricks (LDS past 64 KB),
# 30*31*43 = 39990, 40*40*25 = 40000.  Coordinates stay below 35: the FP32
# distances of both sides are then good to 4e-5 dx, and a candidate more or
# less at the radius adds K(1 - 1e-4) ~ 1e-9.
@pytest.mark.parametrize("bricks", [(31, 24, 22), (30, 31, 43), (40, 40, 25)])
def test_brick_line(ctx, orc, bricks):
    check(ctx, orc, tuple(8 * b - 1 for b in bricks), 20000, 1.0, bricks[0])
