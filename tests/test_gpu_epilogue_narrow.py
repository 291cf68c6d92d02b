"""The FluidSimulation epilogue's workspace on grids a few cells wide, where a
64-cell word holds one short row: what the epilogue adds to a step stays within
its own arrays (two floats a face, the layers, the face lists or the cell words,
whichever are larger)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni", [1, 3, 4])
def test_epilogue_workspace_of_narrow_grids(ni):
    import torch

    import gridfluidsim3d_amd as gf
    dims, dx = (ni, 2000, 2000), 0.1
    pos = np.random.default_rng(1).uniform(0.0, 0.1, size=(100, 3)).astype(np.float32)
    used = []
    for epilogue in (gf.EPILOGUE_NONE, gf.EPILOGUE_FLUIDSIM):
        st = gf.FlipState(pos, np.zeros_like(pos), dims, dx)
        ctx = gf.Context(0)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        ctx.flip_step(st, 1.0 / 120.0, epilogue=epilogue)
        torch.cuda.synchronize()
        used.append(before - torch.cuda.mem_get_info()[0])
        ctx.close()
        del st
    faces = sum(int(np.prod(s)) for s in gf.mac_shapes(dims))
    cells, rows = int(np.prod(dims)), dims[1] * dims[2]
    own = 8 * faces + cells + max(2 * faces, 16 * rows)
    # allocations are whole pages of up to 2 MiB; list offsets per 1024 faces
    assert used[1] - used[0] <= own + 16 * (faces // 1024 + 3) + 6 * (2 << 20), (used, own)
