"""The FluidSimulation epilogue at the edges of its tiles (50x8x8 cells), of
its launches (seven layers) and of its face segments, against the oracle."""
import numpy as np
import pytest

from conftest import NORM_REL_TOL, norm_rel
from test_gpu_epilogue import outside_solid, run_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,layers", [
    ((51, 9, 17), 1), ((50, 8, 8), 7), ((100, 24, 7), 8), ((13, 40, 23), 14), ((120, 3, 16), 15),
    ((1, 30, 2), 100), ((16, 16, 4), 6),
])
def test_epilogue_layers_match_oracle(ctx, orc, dims, layers):
    rng = np.random.default_rng(dims[0] + layers)
    dx, dt = 0.1, 1.0 / 120.0
    ext = np.array(dims) * dx
    # a blob in one corner and single cells, so that layers end inside the grid
    pos = rng.uniform(0.0, 0.35, size=(1500, 3)) * ext
    pos = np.concatenate([pos, (np.array(dims) // 2 + rng.uniform(0.3, 0.7, size=(8, 3))) * dx])
    solid = (rng.uniform(size=dims[::-1]) < 0.06).astype(np.uint8)
    pos = pos.astype(np.float32)
    pos = pos[outside_solid(pos, dx, solid)]
    # smooth velocities: faces reached only at the edge of the radius keep FP32 precision
    vel = np.stack([np.sin(pos[:, 1] + a) for a in range(3)], 1).astype(np.float32)
    got = run_gpu(ctx, pos, vel, dims, dx, dt, 0, 1, solid, layers)
    exp = orc.flip_step_fs(pos, vel, dims, dx, dt, (0.0, -9.8, 0.0), 0.05, 0, solid, layers)
    for key in ("u", "v", "w", "u_old", "v_old", "w_old"):
        assert np.array_equal(got[key] == 0.0, exp[key] == 0.0), key     # the same faces are set
        assert norm_rel(got[key], exp[key]) <= NORM_REL_TOL, key
