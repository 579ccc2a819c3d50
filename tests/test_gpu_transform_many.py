"""GPU parity of the transform adjoint against the FP64 oracle on both sides of
its line between the brick gather, which visits every voxel, and the scatter,
which visits the samples; and of the gather over many grids, whose launches each
take the bricks of the grids that their camera pairs view: grids that end a
launch, grids whose views are split between launches, levels that work-groups
share.

Tolerance: gradients 1e-4 of the largest value, as for the other adjoints.
"""
import numpy as np
import pytest

from oracle import BORDER, LINEAR
from oracle import geometry as G
from oracle import mips as MP
from oracle import resample as R
from test_gpu_transform_gather import cameras, dev, f32, host, ngt_ops, rel  # noqa: F401  (the module's fixture)

pytestmark = pytest.mark.gpu

CLOSE = (1.6, 0.6, 2.6)  # the grid fills about half of the view


def check(ops, cams, dims, out_dhw, C, n, views, levels, mode, seed):
    rng = np.random.default_rng(seed)
    inp = f32(rng.standard_normal((n,) + dims + (C,)))
    g = f32(rng.standard_normal((n, views) + out_dhw + (C,)))
    exp = R.sample_grid_transform_grad(inp, g, *cams, LINEAR, BORDER, R.COORDINATE_MODE[mode], True, "exact",
                                       MP.MIP_LINEAR if levels else MP.MIP_NONE, levels, 0.0)
    got = host(ops.sample_grid_transform_grad(dev(inp), dev(g), *cams, coordinate_mode=mode,
                                              mipmapping="LINEAR" if levels else "NONE", num_mipmaps=levels))
    assert rel(got, exp) < 1e-4


@pytest.mark.parametrize("dims,out_dhw,C,n,views,levels", [
    ((9, 8, 10), (24, 23, 25), 2, 8, 1, 0),      # one launch
    ((9, 8, 10), (24, 23, 25), 4, 17, 1, 0),     # 8 + 8 + 1 grids
    ((9, 8, 10), (24, 23, 25), 4, 3, 5, 0),      # the second grid's views: 3 + 2
    ((9, 8, 10), (24, 23, 25), 4, 1, 17, 0),     # a grid in three launches
    ((70, 66, 65), (24, 23, 22), 4, 1, 2, 0),    # enough bricks for the larger ones
    ((32, 36, 70), (40, 36, 38), 1, 1, 3, 5),
    ((17, 23, 19), (28, 26, 29), 2, 2, 5, 4),    # shared levels in two launches
    ((11, 9, 13), (40, 33, 35), 1, 2, 5, 0),     # the finest level shared, two launches
    ((96, 64, 94), (33, 32, 34), 4, 1, 2, 3),    # level 2 not shared: 4 channels, 144 bricks
    ((11, 9, 13), (18, 17, 19), 1, 1, 2, 1),     # 4.5 cells a voxel: the finest level shared
    ((11, 9, 13), (16, 15, 17), 1, 1, 2, 1),     # 3.2: not shared
    ((9, 8, 10), (5, 4, 6), 1, 17, 1, 0),        # too few values for three launches: scatter
    ((40, 36, 33), (7, 6, 5), 1, 1, 1, 0),       # too few for the voxels
    ((40, 36, 33), (7, 6, 5), 2, 2, 5, 2),
])
def test_adjoint_of_many_grids(ngt_ops, dims, out_dhw, C, n, views, levels):  # noqa: F811
    check(ngt_ops, cameras(dims, out_dhw, views, n, *CLOSE), dims, out_dhw, C, n, views, levels, "TRANSFORM_LINDEPTH",
          300 + n + 7 * C + 3 * views + levels)


@pytest.mark.parametrize("mode", ["TRANSFORM_LINDEPTH", "TRANSFORM"])
@pytest.mark.parametrize("C,levels", [(1, 0), (4, 2)])
def test_camera_close_before_the_grid(ngt_ops, C, levels, mode):  # noqa: F811
    """Bricks next to the camera's plane: corners far outside the view, boxes up to all of it."""
    dims, out_dhw = (16, 12, 20), (26, 22, 24)
    check(ngt_ops, cameras(dims, out_dhw, 3, 1, 0.75, 0.01, 1.6), dims, out_dhw, C, 1, 3, levels, mode, 800 + C)


@pytest.mark.parametrize("dims,out_dhw,C,levels", [
    ((24, 20, 22), (10, 9, 8), 1, 0),    # 0.07 values a voxel: scatter
    ((24, 20, 22), (15, 14, 13), 1, 0),  # 0.26: gather
    ((24, 20, 22), (26, 21, 23), 1, 2),  # 1.2: scatter
    ((24, 20, 22), (30, 26, 24), 1, 2),  # 1.8: gather
    ((24, 20, 22), (15, 14, 13), 4, 2),  # 1.03 with 4 channels: gather
])
def test_adjoint_along_the_axes(ngt_ops, dims, out_dhw, C, levels):  # noqa: F811
    """A grid over the [-1, 1] cube through an orthographic camera of it, as resampling has it."""
    M = G.grid_transform(dims, center=True, scale_=[2.0 / dims[2], 2.0 / dims[1], 2.0 / dims[0]])
    cams = ([G.op_matrix(M).astype(np.float32)], [np.eye(4, dtype=np.float32).reshape(16)],
            [np.eye(4, dtype=np.float32).reshape(16)], [np.asarray([-1, 1, -1, 1, 1, -1], dtype=np.float32)])
    check(ngt_ops, cams, dims, out_dhw, C, 1, 1, levels, "TRANSFORM", 700 + C + levels)
