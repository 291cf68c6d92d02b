"""Point calls where many bricks hold a few points and some hold most: the
sparse bricks' points go straight from memory, behind the others in the sorted
order.  The same bits as the direct kernels, and about the time of the points in
the full bricks."""
import numpy as np
import pytest

from test_gpu_points import DIRECT

pytestmark = pytest.mark.gpu


def uneven(dims, dx, spread, n, box, seed):
    """spread points anywhere (some outside), n in the box of cells."""
    import torch

    import gridfluidsim3d_amd as gf
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rand = lambda m, d: torch.rand((m, 3), generator=g, device="cuda") * torch.tensor(
        d, device="cuda", dtype=torch.float32) * dx
    pos = torch.cat([rand(spread, dims) * 1.02 - 0.01 * dx, rand(n, box)])
    f = [torch.randn(s, generator=g, device="cuda") for s in gf.mac_shapes(dims)]
    return pos[torch.randperm(spread + n, generator=g, device="cuda")].contiguous(), f


# 31 and 32 points a brick on average: sparse ones and others
@pytest.mark.parametrize("dims,spread,n,box", [
    ((80, 72, 64), 22000, 600000, (16, 16, 16)), ((80, 72, 64), 3000, 600000, (8, 8, 8)),
    ((80, 72, 64), 700000, 0, (8, 8, 8)),
])
def test_uneven_same_bits(ctx, dims, spread, n, box):
    import torch
    dx = 0.1
    pos, f = uneven(dims, dx, spread, n, box, spread)
    parts = [pos[s:s + DIRECT].contiguous() for s in range(0, len(pos), DIRECT)]
    got = ctx.g2p_device(pos, *f, dims, dx, 1)
    assert torch.equal(got, torch.cat([ctx.g2p_device(p, *f, dims, dx, 1) for p in parts]))
    for order in (1, 4):
        got = ctx.advect_device(pos, *f, dims, dx, 0.05, order, 1)
        exp = torch.cat([ctx.advect_device(p, *f, dims, dx, 0.05, order, 1) for p in parts])
        assert torch.equal(got, exp)


def test_uneven_linear_same_bits(ctx):
    import torch
    dims, dx = (64, 56, 72), 0.1
    pos, f = uneven(dims, dx, 9000, 1 << 21, (24, 40, 30), 3)
    got = ctx.advect_device(pos, *f, dims, dx, 0.05, 4, 0)
    exp = torch.cat([ctx.advect_device(pos[s:s + DIRECT].contiguous(), *f, dims, dx, 0.05, 4, 0)
                     for s in range(0, len(pos), DIRECT)])
    assert torch.equal(got, exp)


def test_sparse_bricks_cost_little(ctx):
    """Half a million points spread over 33 thousand bricks beside 2.8M in a few:
    a tricubic sample took 3.8 times as long as of 3.3M points in the few when
    each sparse brick had a work-group and an atomic on one word, 1.6 now; 2.5 is
    the bound."""
    import torch
    dims, dx = (256, 256, 256), 0.1

    def best(spread, n):
        pos, f = uneven(dims, dx, spread, n, (256, 40, 40), 1)
        c = (pos / dx).long()
        pos = pos[torch.argsort(c[:, 0] + 256 * (c[:, 1] + 256 * c[:, 2]))].contiguous()
        times = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(3):
                ctx.g2p_device(pos, *f, dims, dx, 1)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)
    both, full = best(500000, 2800000), best(0, 3300000)
    assert both <= 2.5 * full, (both, full)
