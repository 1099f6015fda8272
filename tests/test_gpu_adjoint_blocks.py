"""The adjoint sweep where its blocks of 128 consecutive cells and the rows of
the box do not line up: rows shorter, longer and one off the block, the
smallest extents, a last block that is nearly empty.  Objective, tau, n_s and
u0 gradients against the torch FP64 restatement and its autograd gradient;
tolerances: about 1e-16 per operation over 4 steps of a few hundred, 1e-12 of
the largest value."""
import numpy as np
import pytest
import torch

import iso_reference as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 3, 3), (5, 7, 127), (4, 3, 128), (3, 5, 129), (7, 9, 43), (3, 4, 300)])
def test_gradient_at_block_edges(engine, shape):
    from marbles_amd.adjoint import IsoSolver

    nz, ny, nx = shape
    rng = np.random.default_rng(11)
    ns = torch.tensor(0.1 * rng.random(shape))
    u0 = torch.tensor(0.03 * (rng.random((3,) + shape) - 0.5))
    a, b = ns.clone().requires_grad_(True), u0.clone().requires_grad_(True)
    tau = torch.tensor(0.7, dtype=torch.float64, requires_grad=True)
    J, _ = R.run(shape, a, tau, b, 0.04, 1.0 / 3.0, 4)
    J.backward()
    S = IsoSolver((nx, ny, nz), T0=1.0 / 3.0, u_in=0.04)
    try:
        gJ, gtau, gns, gu0 = S.gradient(ns.cuda(), 0.7, u0.cuda(), 4)
        assert abs(gJ - J.item()) <= 1e-12 * abs(J.item())
        scale = max(abs(tau.grad.item()), a.grad.abs().sum().item())
        assert abs(gtau - tau.grad.item()) <= 1e-12 * scale
        for got, ref in ((gns.cpu(), a.grad), (gu0.cpu(), b.grad)):
            assert (got - ref).abs().max().item() <= 1e-12 * ref.abs().max().item()
    finally:
        S.close()
