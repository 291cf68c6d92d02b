"""The combine of the scatter P2G's tiles by rows and across row ends: grids
whose rows fill the lanes and grids whose rows do not, one and two words of
occupied bricks per row, against the oracle."""
import numpy as np
import pytest

from conftest import NORM_REL_TOL, norm_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [
    (1, 3, 2), (5, 4, 63), (33, 9, 10), (129, 8, 8),    # across row ends
    (250, 10, 12), (64, 200, 3),                        # by rows; u rows of one lane past 64
    (300, 6, 8), (270, 8, 9),                           # two mask words per row of bricks
])
def test_grids_match_oracle(ctx, orc, dims):
    import gridfluidsim3d_amd as gf
    rng = np.random.default_rng(dims[0])
    dx, dt, n = 0.1, 1.0 / 120.0, 6000
    pos = (rng.uniform(-0.01, 1.01, size=(n, 3)) * np.array(dims) * dx).astype(np.float32)
    pos[n // 2:, 0] *= 0.3      # bricks without particles along the rows
    vel = rng.normal(size=(n, 3)).astype(np.float32)
    st = gf.FlipState(pos, vel, dims, dx, keep_old=True, keep_weights=True)
    ctx.flip_step(st, dt, (1.0, -9.8, 0.5), 0.05, gf.TRILINEAR, gf.ORDER_KEEP)
    exp = orc.flip_step(pos, vel, dims, dx, dt, (1.0, -9.8, 0.5), 0.05, 0)
    for c, name in enumerate("uvw"):
        assert norm_rel(st.grid[c].cpu().numpy(), exp[name]) <= NORM_REL_TOL
        off = [0.5 * dx] * 3
        off[c] = 0.0
        nd = gf.mac_shapes(dims)[c][::-1]
        S, W = orc.p2g(pos, vel[:, c].copy(), dx, off, dx, nd)
        assert norm_rel(st.weights[c].cpu().numpy(), W) <= NORM_REL_TOL
        old = np.where(W > 0, S / np.where(W > 0, W, 1), S)
        assert norm_rel(st.grid_old[c].cpu().numpy(), old) <= NORM_REL_TOL
