"""The splat's line between its two sorts for small radii on large grids (few
points take the cell sort) and its gathers by columns and by single nodes: the
same bits on either side, and the time of a call with very few points."""
import numpy as np
import pytest

from conftest import NORM_REL_TOL, norm_rel

pytestmark = pytest.mark.gpu


def splat(ctx, pos, val, dims, dx, radius):
    import torch
    S, W = torch.zeros(dims[::-1], device="cuda"), torch.zeros(dims[::-1], device="cuda")
    ctx.p2g_device(pos, val, radius * dx, (0.0, 0.01, -0.02), dx, dims, S, W)
    return S, W


# a 32nd of the nodes is the line of the cell sort (3.17M nodes, radii of up to a
# cell) and of the sparse gather's longer columns (all)
@pytest.mark.parametrize("dims,radius", [
    ((150, 150, 141), 0.9), ((150, 150, 141), 1.0), ((150, 150, 141), 1.01), ((90, 80, 75), 0.9),
    ((90, 80, 75), 1.7), ((90, 80, 75), 4.0), ((101, 83, 100), 1.0), ((101, 83, 100), 2.5),
])
def test_same_bits_on_both_sides(ctx, orc, dims, radius):
    import torch
    dx = 0.1
    n = -(-int(np.prod(dims)) // 32)
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.0, 1.0, size=(n, 3)) * np.array(dims) * dx
    pos[: n // 2] = rng.uniform(0.3, 0.5, size=(n // 2, 3)) * np.array(dims) * dx
    pos[-1] = -50.0        # reaches no node
    pos, val = pos.astype(np.float32), rng.normal(size=n).astype(np.float32)
    dpos, dval = torch.tensor(pos, device="cuda"), torch.tensor(val, device="cuda")
    S, W = splat(ctx, dpos, dval, dims, dx, radius)
    S1, W1 = splat(ctx, dpos[:-1].contiguous(), dval[:-1].contiguous(), dims, dx, radius)
    assert torch.equal(S, S1) and torch.equal(W, W1)
    Se, We = orc.p2g(pos, val, radius * dx, (0.0, 0.01, -0.02), dx, dims)
    assert norm_rel(S.cpu().numpy(), Se) <= NORM_REL_TOL
    assert norm_rel(W.cpu().numpy(), We) <= NORM_REL_TOL


# single nodes and columns of several: the same points on a taller grid
@pytest.mark.parametrize("radius", [1.0, 2.5, 4.0])
@pytest.mark.parametrize("n", [40000, 900000])
def test_columns_and_single_nodes_same_bits(ctx, n, radius):
    import torch
    dx = 0.1
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    pos = torch.rand((n, 3), generator=g, device="cuda") * 3.0
    val = torch.randn(n, generator=g, device="cuda")
    S, W = splat(ctx, pos, val, (40, 40, 40), dx, radius)
    S1, W1 = splat(ctx, pos, val, (40, 40, 800), dx, radius)
    assert torch.equal(S, S1[:40]) and torch.equal(W, W1[:40])


def test_very_few_points_cost_what_the_cell_sort_costs(ctx):
    """100 points on 100^3 nodes: just above four cells' radius the cell sort
    always took them; at four the bricks took twice as long, and half as long
    again is the bound."""
    import torch
    dims, dx = (100, 100, 100), 0.1
    pos = torch.rand((100, 3), device="cuda") * 10.0
    val = torch.randn(100, device="cuda")
    S, W = torch.zeros(dims, device="cuda"), torch.zeros(dims, device="cuda")

    def best(radius):
        times = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                ctx.p2g_device(pos, val, radius * dx, (0.0, 0.0, 0.0), dx, dims, S, W)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)
    at, above = best(4.0), best(4.01)
    assert at <= 1.5 * above, (at, above)
