"""The advection adjoint with bricks 4, 8 and 16 cells deep, which it takes by how
many of them there are: 24 instances in one call run the deepest, 12 the middle
ones, and each instance alone the flattest: the same gradients.

Tolerance: where every corner stays in a tile the fp32 tile partials differ in
rounding (at most 8 per cell, and twice: 16 * 2^-24 < 1e-6); where corners leave
them, up to 64 fp32 additions per cell in no fixed order come on top, 4e-6: 1e-5.
"""
import numpy as np
import pytest

import test_gpu_advect_bricks as TB
from test_gpu_advect_bricks import ngt_ops  # noqa: F401  (the module's fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vmax,tol", [(1.9, 1e-6), (6.0, 1e-5)])
@pytest.mark.parametrize("C,boundary", [(1, "BORDER"), (3, "BORDER"), (2, "CLAMP"), (4, "WRAP")])
def test_depths_agree(ngt_ops, C, boundary, vmax, tol):  # noqa: F811
    rng = np.random.default_rng(90 + C + int(vmax))
    N, shape = 24, (37, 20, 70)
    cases = [TB._case_inputs(rng, shape, C, False, vmax=vmax) for _ in range(N)]
    rho, vel = (TB.dev(np.stack([c[i] for c in cases])) for i in (0, 2))
    g = TB.dev(rng.standard_normal((N, 1) + shape + (C,)))

    def grads(sl):
        d, v = (t[sl].clone().requires_grad_() for t in (rho, vel))
        ngt_ops.advect_grid_semi_langrange(d, v, timestep=-1.0, order=2, clamp_extrema="MC_SMOOTH", boundary=boundary,
                                           separate_velocity_batch=False).backward(g[sl])
        return TB.host(d.grad), TB.host(v.grad)

    deep, middle = grads(slice(0, N)), grads(slice(0, 12))
    for n in (0, 7, 11, 23):
        flat = grads(slice(n, n + 1))
        for got, exp in zip(deep, flat):
            assert TB.rel(got[n:n + 1], exp) < tol
        if n < 12:
            for got, exp in zip(middle, flat):
                assert TB.rel(got[n:n + 1], exp) < tol
