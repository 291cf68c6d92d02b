"""A recorded step whose tape arrays start on any 4-byte address, as the header
allows: the same tape, and the same gradient, as with torch's own arrays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_tape_on_any_address(ctx, monkeypatch, shift):
    import torch

    from gridfluidsim3d_amd import gfsx
    dims, dx, dt, n = (33, 24, 20), 0.1, 1.0 / 120.0, 5001
    rng = np.random.default_rng(shift)
    ext = np.array(dims)[:, None] * dx
    dev = lambda a: torch.tensor(a.astype(np.float32), device="cuda")
    x, v = dev(rng.uniform(-0.02, 1.02, size=(3, n)) * ext), dev(rng.normal(size=(3, n)))
    a, b = dev(rng.normal(size=(3, n))), dev(rng.normal(size=(3, n)))

    class Shifted(gfsx.FlipTape):
        def __init__(self, n, dims, starts, device):
            super().__init__(n, dims, starts, device)
            i32, f32 = torch.int32, torch.float32
            self.perm = torch.empty(n + 4, dtype=i32, device=device)[shift:shift + n]
            self.start = torch.empty(starts + 4, dtype=i32, device=device)[shift:shift + starts]
            self.xs = [torch.empty(n + 4, dtype=f32, device=device)[shift:shift + n]
                       for _ in range(3)]

    def record():
        x1, v1, tape = ctx.flip_step_record(x, v, dims, dx, dt)
        gx, gv = ctx.flip_step_backward(x, v, a, b, dims, dx, dt, tape=tape)
        return [x1, v1, tape.perm, tape.start, *tape.xs, gx, gv]
    want = record()
    monkeypatch.setattr(gfsx, "FlipTape", Shifted)
    got = record()
    assert got[3].data_ptr() % 16 == 4 * shift
    for p, q in zip(got, want):
        assert torch.equal(p, q)
