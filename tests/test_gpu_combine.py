"""The combine of the scatter P2G's tiles by rows and across row ends.  A
scene alone takes one of the two by its own rows; in a batch all scenes take
one by the rows of all.  Either way a scene's results are the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS = [(250, 10, 12), (300, 6, 8)]    # fill their lanes (300: two mask words a row)
ENDS = [(1, 3, 2), (5, 4, 63), (33, 9, 10), (129, 8, 8), (64, 200, 3), (270, 8, 9)]


def state(dims, seed, n=6000):
    import gridfluidsim3d_amd as gf
    rng = np.random.default_rng(seed)
    pos = (rng.uniform(-0.01, 1.01, size=(n, 3)) * np.array(dims) * 0.1).astype(np.float32)
    pos[n // 2:, 0] *= 0.3      # bricks without particles along the rows
    vel = rng.normal(size=(n, 3)).astype(np.float32)
    return gf.FlipState(pos, vel, dims, 0.1, keep_old=True, keep_weights=True)


@pytest.mark.parametrize("filler,scenes", [((40, 40, 40), ROWS + ENDS), ((256, 90, 90), ENDS)])
def test_combine_same_bits_alone_and_batched(ctx, filler, scenes):
    """The filler's faces decide for the batch: across row ends, by rows."""
    import torch
    batch = [state(d, i) for i, d in enumerate(scenes)] + [state(filler, 99)]
    kw = dict(dt=1.0 / 120.0, body_force=(1.0, -9.8, 0.5))
    ctx.flip_step_batched(batch, **kw)
    for i, d in enumerate(scenes):
        one = state(d, i)
        ctx.flip_step(one, **kw)
        for a, b in ((one.grid, batch[i].grid), (one.grid_old, batch[i].grid_old),
                     (one.weights, batch[i].weights), (one.cur_x, batch[i].cur_x)):
            for p, q in zip(a, b):
                assert torch.equal(p, q)
        assert all(bool(w.abs().sum() > 0) for w in one.weights)
