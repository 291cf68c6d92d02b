"""gfsx_remove_particles at the sizes where a cell changes from one wave to
one work-group, and at block ends of the compaction, against a numpy
selection by key."""
import numpy as np
import pytest

from test_gpu_removal import _splitmix_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap,extra", [(1, 0), (63, 1), (64, 1023), (255, 1024), (256, 1025),
                                       (300, 7)])
def test_removal_cell_sizes(ctx, cap, extra):
    import gridfluidsim3d_amd as gf
    dims, dx, seed = (12, 5, 3), 0.25, 77
    lens = [0, 1, 2, 63, 64, 65, 127, 128, 255, 256, 257, 258, 511, 513, cap, cap + 1, 1025]
    rng = np.random.default_rng(cap)
    cells = rng.permutation(12 * 5 * 3)[:len(lens) + 2]
    solid = np.zeros((3, 5, 12), np.uint8)
    members = [np.full(m, c) for m, c in zip(lens, cells)]
    for c, m in zip(cells[-2:], (40, 700)):      # solid cells lose all, whatever their count
        solid.reshape(-1)[c] = 1
        members.append(np.full(m, c))
    flat = rng.permutation(np.concatenate(members + [np.full(extra, -1)]))
    pos = np.empty((flat.size, 3), np.float32)
    f = rng.uniform(0.1, 0.9, size=pos.shape)
    pos[:, 0] = (flat % 12 + f[:, 0]) * dx
    pos[:, 1] = (flat // 12 % 5 + f[:, 1]) * dx
    pos[:, 2] = (flat // 60 + f[:, 2]) * dx
    pos[flat < 0] = -1.0                         # outside the grid: kept
    vel = rng.normal(size=pos.shape).astype(np.float32)
    keys = _splitmix_np(seed, np.arange(flat.size))
    keep = np.ones(flat.size, bool)
    for c in cells:
        m = np.flatnonzero(flat == c)
        if solid.reshape(-1)[c]:
            keep[m] = False
        elif m.size > cap:
            keep[m] = False
            keep[m[np.argsort(keys[m])[:cap]]] = True
    st = gf.FlipState(pos, vel, dims, dx, track_ids=True, solid=solid)
    assert ctx.remove_particles(st, cap, seed) == keep.sum()
    assert np.array_equal(st.particle_ids().cpu().numpy(), np.flatnonzero(keep))
    assert np.array_equal(st.positions().cpu().numpy(), pos[keep])
    assert np.array_equal(st.velocities().cpu().numpy(), vel[keep])
