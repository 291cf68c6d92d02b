"""The scan of the brick sort's bin counts and the step's work lists at the
edges of their launches: one tile of 1024 bins and one bin more, 16 and 17
tiles (work-groups adding up counts, or tile sums), 32 thousand bins and more
(one or four bins a thread), more than 8192 tiles (tile sums scanned first).
The sorted order is exact against numpy's stable argsort, and the step's fields
and particles have the bits of the 4-cell G2P bricks, which use no list."""
import numpy as np
import pytest

from test_gpu_brick import brick_keys

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [
    (8, 8, 8), (56, 72, 16), (64, 64, 16), (120, 128, 64), (128, 128, 64), (136, 136, 112),
    (128, 128, 128), (136, 128, 120), (816, 816, 808),
])
def test_starts_and_lists(ctx, dims):
    import torch

    import gridfluidsim3d_amd as gf
    print("[bins] %s" % (dims,), flush=True)
    rng = np.random.default_rng(dims[0])
    n = 30000
    pos = (rng.uniform(-0.02, 1.02, size=(n, 3)) * np.array(dims) * 0.1).astype(np.float32)
    pos[: n // 8] = rng.uniform(0.0, 0.8, size=(n // 8, 3))
    vel = rng.normal(size=(n, 3)).astype(np.float32)
    out = []
    try:
        for edge in (8, 4):
            ctx.set_option("g2p_brick", edge)
            st = gf.FlipState(pos, vel, dims, 0.1, track_ids=True)
            ctx.flip_step(st, 1.0 / 120.0, order=gf.ORDER_SORTED)
            out.append(list(st.cur_x + st.cur_v) + [st.particle_ids()])
            del st
    finally:
        ctx.set_option("g2p_brick", 8)
    for a, b in zip(*out):
        assert torch.equal(a, b)
    ids = out[0][-1].cpu().numpy().astype(np.int64)
    assert np.array_equal(ids, np.argsort(brick_keys(pos, dims, 0.1), kind="stable"))
