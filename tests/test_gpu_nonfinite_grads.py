"""A gradient that is no finite number stays where it belongs in the advection
adjoint: with no displacement every sample lies on its own cell, whose upper
trilinear weights are 0, so the density gradient is the output gradient and a
NaN or infinity in it reaches no other cell.

Tolerance: the other cells' gradients are sums of one value with zeros, halved
and added back exactly: equal.
"""
import numpy as np
import pytest
import torch

from test_gpu_advect_bricks import dev, ngt_ops  # noqa: F401  (the module's fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("C,order", [(1, 1), (1, 2), (3, 1), (3, 2)])
def test_nonfinite_gradient_keeps_to_its_cell(ngt_ops, C, order, bad):  # noqa: F811
    shape = (9, 10, 35)
    rng = np.random.default_rng(11 + C + order)
    rho = dev(rng.uniform(0.5, 1.0, (1,) + shape + (C,))).requires_grad_()
    vel = torch.zeros((1,) + shape + (3,), device="cuda:0", requires_grad=True)
    g = dev(rng.standard_normal((1, 1) + shape + (C,)))
    for cell in ((4, 3, 5), (7, 8, 32)):  # inside a brick, and in its neighbour's halo
        g[(0, 0) + cell] = bad
    out = ngt_ops.advect_grid_semi_langrange(rho, vel, timestep=-1.0, order=order, clamp_extrema="NONE",
                                             boundary="BORDER", separate_velocity_batch=False)
    out.backward(g)
    ok = torch.isfinite(g[0])
    assert torch.equal(torch.isfinite(rho.grad), ok)
    assert torch.equal(rho.grad[ok], g[0][ok])
