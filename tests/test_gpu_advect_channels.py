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
