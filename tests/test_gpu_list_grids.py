"""The grids of steps whose scatter takes its bricks from the work lists, at the
lists' own lines, against the FP64 oracle, which knows no bricks: a bin missing,
listed twice or wrongly cleared shows in the weights, the sums or the fluid
mask.  (Comparing two brick sizes of G2P cannot show it: both scatter from the
same list.)

Weights W, sums S = n W and the body force's increments are compared norm-wise:
n alone divides by weights near zero.  FP32 distances leave K good to 1e-6 or
so of its maximum, W and S are exact sums of such terms, and the increments are
0.08 beside velocities of about 4 (rounding 5e-7 / 0.08): NORM_REL_TOL."""
import numpy as np
import pytest

from conftest import NORM_REL_TOL, norm_rel

pytestmark = pytest.mark.gpu


# bins are 8 per 8^3 cells and one: 9, 1025, 17 tiles of 1024 and 16, either side of
# 32768, where a thread takes four bins instead of one
@pytest.mark.parametrize("dims,n", [
    ((8, 8, 8), 257), ((64, 64, 16), 1500), ((100, 90, 7), 1200), ((64, 64, 256), 30000),
    ((64, 72, 216), 30000), ((120, 128, 128), 60000), ((128, 128, 128), 60000),
    ((136, 128, 128), 2000),
])
def test_listed_bricks_give_the_oracles_grids(ctx, orc64, dims, n):
    import torch

    import gridfluidsim3d_amd as gf
    rng = np.random.default_rng(dims[0] + n)
    dx, dt, bf = 0.125, 1.0 / 120.0, (9.8, -9.8, 9.8)
    pos = rng.uniform(-0.02, 1.02, size=(n, 3)) * np.array(dims) * dx
    pos[: n // 4] = rng.uniform(0.1, 0.9, size=(n // 4, 3))      # a quarter in one brick
    pos, vel = pos.astype(np.float32), rng.normal(size=(n, 3)).astype(np.float32)
    want = orc64.flip_step(pos, vel, dims, dx, dt, bf, 0.05)
    st = gf.FlipState(pos, vel, dims, dx, keep_old=True, keep_weights=True)
    ctx.flip_step(st, dt, bf, 0.05, gf.TRILINEAR, gf.ORDER_SORTED)
    torch.cuda.synchronize()
    for c, k in enumerate("uvw"):
        W, W64 = st.weights[c].cpu().numpy().astype(np.float64), want["w" + k]
        old = st.grid_old[c].cpu().numpy().astype(np.float64)
        assert norm_rel(W, W64) <= NORM_REL_TOL, k
        assert norm_rel(old * W, want[k + "_old"] * W64) <= NORM_REL_TOL, k
        force = st.grid[c].cpu().numpy() - old
        assert norm_rel(force, want[k] - want[k + "_old"]) <= NORM_REL_TOL, k
