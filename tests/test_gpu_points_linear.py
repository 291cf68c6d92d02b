"""The trilinear Runge-Kutta steps by bricks (order 4 from 2^21 points on,
order 3 from 2^22), in FP64 cells as well as where 1/dx is a power of two, on either side of
that line: the same bits as the direct kernels, which a call of few points
takes."""
import numpy as np
import pytest

from test_gpu_points import DIRECT, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,line", [(3, 1 << 22), (4, 1 << 21)])
@pytest.mark.parametrize("dims,dx,more,speed", [
    ((40, 33, 27), 0.1, 0, 1.0),
    ((40, 33, 27), 0.1, -1, 1.0),
    ((40, 33, 27), 0.1, 2851, 20.0),         # stages that leave the boxes
    ((33, 40, 9), 0.125, 0, 2.0),
])
def test_linear_steps_same_bits_as_direct(ctx, dims, dx, more, speed, order, line):
    import torch
    n = line + more
    _, _, (pos, u, v, w) = scene(dims, dx, n, speed, order)
    got = ctx.advect_device(pos, u, v, w, dims, dx, 0.01, order, 0)
    exp = torch.cat([ctx.advect_device(pos[s:s + DIRECT].contiguous(), u, v, w, dims, dx, 0.01,
                                       order, 0) for s in range(0, n, DIRECT)])
    nan = torch.isnan(exp)
    assert torch.equal(nan, torch.isnan(got))
    assert torch.equal(got[~nan].view(torch.int32), exp[~nan].view(torch.int32))
