"""GPU parity of the brick-tiled advection adjoint with 3 and 4 channels (the
velocity self-advection and the light-and-density grids), whose channels take
turns in one LDS tile, against the FP64 oracle on grids of several bricks.

Tolerances as for 1 and 2 channels (test_gpu_advect_bricks.py): forward 1e-5
and gradients 1e-4 of the largest value.
"""
import numpy as np
import pytest
import torch

from oracle import BORDER, CLAMP, WRAP
from oracle import advect as A

import test_gpu_advect_bricks as TB
from test_gpu_advect_bricks import ngt_ops  # noqa: F401  (the module's fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,shape", [(3, (34, 17, 37)), (4, (33, 9, 12)), (3, (7, 5, 70))])
@pytest.mark.parametrize("order,clamp,bound,staggered,vmax", [
    (2, "MC_SMOOTH", BORDER, False, 1.9), (2, "MC_SMOOTH", BORDER, True, 3.5), (2, "NEGATIVE", CLAMP, False, 1.9),
    (1, "NEGATIVE", WRAP, True, 1.9), (1, "NONE", BORDER, False, 3.5)])
def test_advect_channels_across_bricks(ngt_ops, C, shape, order, clamp, bound, staggered, vmax):  # noqa: F811
    rng = np.random.default_rng(2000 + 31 * C + 7 * order + bound + int(10 * vmax) + shape[0])
    rho, faces, vc = TB._case_inputs(rng, shape, C, staggered, vmax=vmax)
    exp = A.warp_forward(rho, vc, 1.0, order, clamp, bound)
    rt = TB.dev(rho[None]).requires_grad_()
    vel = TB._vel_leaves(faces, vc)
    out = ngt_ops.advect_grid_semi_langrange(rt, vel, timestep=-1.0, order=order, clamp_extrema=clamp,
                                             boundary=TB.BNAME[bound], separate_velocity_batch=False)
    assert TB.rel(TB.host(out)[0, 0], exp) < TB.FWD_TOL
    g = TB.f32(rng.standard_normal(exp.shape))
    out.backward(TB.dev(g[None, None]))
    vel_np = tuple(TB.dev(f[None]) for f in faces) if staggered else TB.dev(vc[None])
    gpu = TB._gpu_parts(ngt_ops, TB.dev(rho[None]), vel_np, order, clamp, bound, out)
    TB._check_grads(rt, vel, faces, rho, vc, g, order, clamp, bound, gpu)


@pytest.mark.parametrize("C", [1, 3])
def test_advect_deep_bricks_equal_flat_ones(ngt_ops, C):  # noqa: F811
    """Twelve instances in one call fill the GPU with 8-cell-deep bricks, each
    alone runs 4-cell-deep ones: the same gradients up to the rounding of the
    fp32 tile partials (at most 8 per cell, and twice: 16 * 2^-24 < 1e-6)."""
    rng = np.random.default_rng(77 + C)
    N, shape = 12, (37, 20, 70)
    rho = [TB._case_inputs(rng, shape, C, False, vmax=1.9) for _ in range(N)]
    dens = TB.dev(np.stack([r[0] for r in rho])).requires_grad_()
    vel = TB.dev(np.stack([r[2] for r in rho])).requires_grad_()
    g = TB.dev(rng.standard_normal((N, 1) + shape + (C,)))
    args = dict(timestep=-1.0, order=2, clamp_extrema="MC_SMOOTH", boundary="BORDER", separate_velocity_batch=False)
    ngt_ops.advect_grid_semi_langrange(dens, vel, **args).backward(g)
    for n in range(0, N, 5):
        d, v = (t.detach()[n:n + 1].clone().requires_grad_() for t in (dens, vel))
        ngt_ops.advect_grid_semi_langrange(d, v, **args).backward(g[n:n + 1])
        assert TB.rel(TB.host(dens.grad)[n:n + 1], TB.host(d.grad)) < 1e-6
        assert TB.rel(TB.host(vel.grad)[n:n + 1], TB.host(v.grad)) < 1e-6
