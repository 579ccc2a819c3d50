"""GPU parity of the ray adjoint's gather of two and four channels against the
scatter adjoint of the same samples, on grids that take bricks of 8^3 and of
16 x 8 x 8 cells (2048 of them), off their extents, in every blend mode.

Tolerance: gradients 1e-4 of the largest value, as for the other adjoints.
"""
import numpy as np
import pytest

from test_gpu_raymarch_gather import cameras, dev, ngt_ops, rel  # noqa: F401  (the module's fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(121, 130, 113), (17, 30, 41)])
@pytest.mark.parametrize("C", [2, 4])
@pytest.mark.parametrize("blend", ["BEER_LAMBERT", "ALPHA", "ALPHA_ADDITIVE", "ADDITIVE"])
def test_channels_match_scatter(ngt_ops, monkeypatch, dims, C, blend):  # noqa: F811
    out_dhw = (45, 21, 30)
    rng = np.random.default_rng(8200 + sum(dims) + C)
    cams = cameras(dims, out_dhw, 3, 30.0)
    x = dev(rng.uniform(0.0, 0.05, (1,) + dims + (C,)))
    out = ngt_ops.raymarch_grid_transform(x, *cams, out_dhw, blending_mode=blend)
    g = dev(rng.standard_normal(tuple(out.shape)))
    got = ngt_ops.raymarch_grid_transform_grad(x, out, g, *cams, out_dhw, blending_mode=blend)
    monkeypatch.setattr(ngt_ops, "use_gather_adjoint", False)
    scatter = ngt_ops.raymarch_grid_transform_grad(x, out, g, *cams, out_dhw, blending_mode=blend)
    assert rel(got, scatter.cpu().double().numpy()) < 1e-4
