"""The rollout's gradient where faces take little weight.

Sparse particles leave faces that one of them touches at the rim of the kernel
(W down to 1e-10): the P2G adjoint divides by W there, so another rounding of
its distances, of dL/dg + dL/dn or of its sums gives other entries, by up to
7e-5 of the largest in these scenes.  golden/rollout_gradient.npz holds two
scenes of 1500 particles on 24x21x19 cells, dx = 1/24, and the gradient of the
density loss (target 0, three steps of 1/240 s) by the initial velocities, as
the step's adjoint gave it on an MI355X with a sum each for dL/dg and dL/dn,
x^2 of the squared distance unrounded, and particle sums added once.
"""
import os

import numpy as np
import pytest
import torch

import gridfluidsim3d_amd as gf
from gridfluidsim3d_amd import autograd as gfa

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "rollout_gradient.npz")
# of the largest entry: the adjoint's own tolerance against FP64 (test_gpu_adjoint.py)
TOL = 2e-5


@pytest.mark.parametrize("tape", [True, False])
@pytest.mark.parametrize("scene", [0, 1])
def test_gradient_on_faces_of_little_weight(scene, tape):
    data = np.load(GOLDEN)
    dims, dx = (24, 21, 19), 1.0 / 24.0
    ctx = gf.Context(0)
    x0 = torch.tensor(data["x%d" % scene], device="cuda")
    v0 = torch.tensor(data["v%d" % scene], device="cuda").requires_grad_(True)
    x, _ = gfa.rollout(ctx, x0, v0, dims, dx, 3, 1.0 / 240.0, tape=tape)
    loss = gfa.density_loss(ctx, x, torch.zeros(dims[::-1], device="cuda"), dims, dx)
    (grad,) = torch.autograd.grad(loss, v0)
    want = data["grad%d" % scene].astype(np.float64)
    err = np.abs(grad.cpu().numpy() - want).max() / np.abs(want).max()
    assert err <= TOL, err
    ctx.close()
