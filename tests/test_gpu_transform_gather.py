"""GPU parity of the transform adjoint's brick gather (LINEAR, BORDER, forward
modes) against the FP64 oracle: extents off the brick sizes and of one cell,
more camera pairs than one launch takes, mips, cameras inside the grid (whose
bricks project behind the camera), and a singular model matrix, which scatters.

Tolerance: gradients 1e-4 of the largest value, as for the scatter.
"""
import numpy as np
import pytest
import torch

from oracle import BORDER, LINEAR
from oracle import geometry as G
from oracle import mips as MP
from oracle import resample as R

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ngt_ops():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from ngt import ops, _lib
    _lib.load()
    return ops


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a, dtype=np.float32))).to("cuda:0")


def host(t):
    return t.detach().cpu().double().numpy()


def f32(a):
    return np.asarray(a, dtype=np.float32).astype(np.float64)


def rel(got, exp):
    return float(np.max(np.abs(got - exp))) / max(float(np.max(np.abs(exp))), 1e-30)


def cameras(dims, out_dhw, views, n, dist, near, far):
    """n grids, each shifted by its own fraction of a cell, before ring cameras."""
    Ms = [G.op_matrix(G.grid_transform(dims, translation_=(0.0123 + 0.05 * i, -0.0217, 0.0311), center=True,
                                       scale_=[1.0 / max(dims)] * 3)).astype(np.float32) for i in range(n)]
    cams = G.look_at_ring_cameras(views, dist, 50.0, out_dhw[2] / out_dhw[1], near, far)
    return (Ms, [G.op_matrix(c[0]).astype(np.float32) for c in cams],
            [G.op_matrix(c[1]).astype(np.float32) for c in cams], [c[2].astype(np.float32) for c in cams])


@pytest.mark.parametrize("dims,out_dhw,C,n,views,mip,ring", [
    ((9, 17, 13), (11, 7, 10), 4, 1, 3, MP.MIP_NONE, (3.0, 2.0, 4.0)),
    ((9, 17, 13), (11, 7, 10), 2, 3, 4, MP.MIP_NONE, (3.0, 2.0, 4.0)),    # 12 pairs: two launches
    ((18, 8, 33), (9, 5, 6), 1, 2, 5, MP.MIP_LINEAR, (3.0, 2.0, 4.0)),    # 10 pairs, coarse cells: all levels
    ((18, 9, 33), (9, 5, 6), 4, 1, 2, MP.MIP_LINEAR, (3.0, 2.0, 4.0)),
    ((16, 12, 20), (13, 9, 12), 1, 1, 3, MP.MIP_NONE, (0.2, 0.05, 1.2)),  # cameras inside the grid
    ((16, 12, 20), (13, 9, 12), 2, 1, 2, MP.MIP_LINEAR, (0.2, 0.05, 1.2)),
    ((1, 12, 7), (9, 6, 8), 1, 1, 3, MP.MIP_NONE, (3.0, 2.0, 4.0)),
    ((70, 66, 65), (7, 6, 5), 1, 1, 2, MP.MIP_NONE, (3.0, 2.0, 4.0)),     # enough bricks for the larger ones
])
@pytest.mark.parametrize("mode", ["TRANSFORM_LINDEPTH", "TRANSFORM"])
def test_gather_adjoint(ngt_ops, dims, out_dhw, C, n, views, mip, ring, mode):
    rng = np.random.default_rng(900 + dims[0] + 7 * C + 3 * views + mip)
    levels = 0 if mip == MP.MIP_NONE else 3
    cams = cameras(dims, out_dhw, views, n, *ring)
    inp = f32(rng.standard_normal((n,) + dims + (C,)))
    g = f32(rng.standard_normal((n, views) + out_dhw + (C,)))
    exp = R.sample_grid_transform_grad(inp, g, *cams, LINEAR, BORDER, R.COORDINATE_MODE[mode], True, "exact", mip,
                                       levels, 0.0)
    got = host(ngt_ops.sample_grid_transform_grad(dev(inp), dev(g), *cams, coordinate_mode=mode,
                                                  mipmapping="NONE" if mip == MP.MIP_NONE else "LINEAR",
                                                  num_mipmaps=levels))
    assert rel(got, exp) < 1e-4


def test_singular_model_matrix(ngt_ops):
    """A model matrix without an inverse (taken as 0) puts every sample on the
    grid's corner, q = -0.5 on each axis: an eighth of every gradient there."""
    rng = np.random.default_rng(5)
    dims, out_dhw = (6, 5, 7), (4, 3, 5)
    M, V, P, F = cameras(dims, out_dhw, 2, 1, 3.0, 2.0, 4.0)
    M = [np.zeros(16, np.float32)]
    g = f32(rng.standard_normal((1, 2) + out_dhw + (1,)))
    got = host(ngt_ops.sample_grid_transform_grad(dev(rng.standard_normal((1,) + dims + (1,))), dev(g), M, V, P, F))
    exp = np.zeros_like(got)
    exp[0, 0, 0, 0, 0] = 0.125 * g.sum()
    assert rel(got, exp) < 1e-4
