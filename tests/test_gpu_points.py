"""Point samples and Runge-Kutta steps gathered by grid brick
(gfsx_points.hip): the same bits as the direct kernels, which a call of few
points takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIRECT = 60000   # points of a call that samples straight from memory


def scene(dims, dx, n, speed, seed):
    import torch

    import gridfluidsim3d_amd as gf
    rng = np.random.default_rng(seed)
    ext = np.array(dims) * dx
    pos = rng.uniform(-0.02, 1.02, size=(n, 3)) * ext
    # a crowded corner, cell faces, and values with no cell
    pos[: n // 3] *= 0.2
    pos[-400:] = np.round(pos[-400:] / dx) * dx
    pos[7] = np.nan
    pos[11, 1] = np.inf
    pos[13] = ext
    pos[17] = 0.0
    pos = pos[rng.permutation(n)].astype(np.float32)
    fields = [(speed * rng.normal(size=s)).astype(np.float32) for s in gf.mac_shapes(dims)]
    return pos, fields, [torch.tensor(a, device="cuda") for a in [pos] + fields]


@pytest.mark.parametrize("stencil", [0, 1])
@pytest.mark.parametrize("dims,dx,n,speed", [
    ((16, 8, 24), 0.125, 200000, 0.5),       # whole bricks, the smallest call of the path
    ((17, 9, 31), 0.1, 530001, 1.0),         # ragged bricks, FP64 cells
    ((64, 40, 33), 0.0625, 1048601, 9.0),    # stages that leave the boxes
    ((257, 250, 255), 0.03125, 3300007, 1.0),   # nearly empty bricks, many histogram words
])
def test_points_same_bits_as_direct(ctx, dims, dx, n, speed, stencil):
    import torch
    pos, fields, (dpos, u, v, w) = scene(dims, dx, n, speed, 5)
    parts = [dpos[s:s + DIRECT].contiguous() for s in range(0, n, DIRECT)]

    def same(a, b):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    out = ctx.g2p_device(dpos, u, v, w, dims, dx, stencil)
    same(out, torch.cat([ctx.g2p_device(p, u, v, w, dims, dx, stencil) for p in parts]))
    for order in (1, 2, 3, 4):
        got = ctx.advect_device(dpos, u, v, w, dims, dx, 0.01, order, stencil)
        exp = torch.cat([ctx.advect_device(p, u, v, w, dims, dx, 0.01, order, stencil)
                         for p in parts])
        nan = torch.isnan(exp)
        assert torch.equal(nan, torch.isnan(got))
        same(got[~nan], exp[~nan])
    # in place, as the reference's overload (particleadvector.cpp:457-465)
    inp = dpos.clone()
    ctx.g2p_device(inp, u, v, w, dims, dx, stencil, out=inp)
    same(inp, out)


def test_points_on_two_streams(ctx):
    """Calls that share the context's workspace from two streams."""
    import torch
    dims, dx, n = (40, 40, 40), 0.05, 530000
    _, _, (a, u, v, w) = scene(dims, dx, n, 1.0, 8)
    _, _, (b, _, _, _) = scene(dims, dx, n + 70000, 1.0, 9)
    exp = [torch.cat([ctx.g2p_device(p[s:s + DIRECT].contiguous(), u, v, w, dims, dx, 1)
                      for s in range(0, p.shape[0], DIRECT)]) for p in (a, b)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for _ in range(3):
        got = []
        for st, p in zip(streams, (a, b)):
            with torch.cuda.stream(st):
                got.append(ctx.g2p_device(p, u, v, w, dims, dx, 1))
        torch.cuda.synchronize()
        for g, e in zip(got, exp):
            assert torch.equal(g, e)
