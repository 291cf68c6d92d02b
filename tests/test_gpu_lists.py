"""The work lists of the brick step: shares of crowded G2P bricks, steps of
far fewer particles than bins and of far more, against the 4-cell G2P bricks
(which take every bin, listed or not): the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,n", [
    ((64, 64, 64), 1), ((64, 64, 64), 0), ((100, 90, 7), 1200), ((64, 64, 64), 1025),
    ((8, 8, 8), 255), ((8, 8, 8), 256), ((8, 8, 8), 257), ((9, 8, 8), 5000),
    ((16, 24, 8), 1300000),
])
@pytest.mark.parametrize("order", [0, 1])
def test_lists_same_bits(ctx, dims, n, order):
    import torch

    import gridfluidsim3d_amd as gf
    rng = np.random.default_rng(n + dims[0])
    pos = rng.uniform(-0.3, 1.3, size=(n, 3)) * np.array(dims) * 0.1
    pos[: n // 2] = np.clip(pos[: n // 2], 0.05, 0.75)      # half of them in one brick
    vel = rng.normal(size=(n, 3))
    out = []
    try:
        for edge in (8, 4):
            ctx.set_option("g2p_brick", edge)
            st = gf.FlipState(pos.astype(np.float32), vel.astype(np.float32), dims, 0.1,
                              track_ids=True)
            for _ in range(2):
                ctx.flip_step(st, 1.0 / 120.0, order=order)
            out.append(st.cur_x + st.cur_v + st.grid + [st.particle_ids()])
    finally:
        ctx.set_option("g2p_brick", 8)
    for a, b in zip(*out):
        assert torch.equal(a, b)
