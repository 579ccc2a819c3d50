"""GPU parity of the transform adjoint's coarse levels, whose bricks share their
candidates among several work-groups (4, 32 and 256 at the first split level, the
next and the coarser ones), against the FP64 oracle: pyramids down to single cells, several grids, more
pairs than one launch takes, and cells coarse enough that every level is read.

Tolerance: gradients 1e-4 of the largest value, as for the scatter.
"""
import numpy as np
import pytest

from oracle import BORDER, LINEAR
from oracle import mips as MP
from oracle import resample as R

from test_gpu_transform_gather import cameras, dev, f32, host, ngt_ops, rel  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,out_dhw,C,n,views,levels", [
    ((32, 36, 70), (13, 9, 11), 1, 1, 3, 5),
    ((32, 40, 33), (5, 4, 6), 4, 1, 2, 5),
    ((17, 23, 19), (3, 3, 4), 2, 2, 5, 4),   # 10 pairs: two launches
    ((20, 16, 16), (40, 33, 35), 1, 1, 2, 2),
    ((11, 9, 13), (40, 33, 35), 2, 1, 2, 2),  # every level split: 31 cells of a view to a voxel
    ((11, 9, 13), (40, 33, 35), 1, 2, 5, 0),  # the finest alone, 10 pairs: two launches
    ((96, 64, 94), (7, 6, 5), 4, 1, 2, 3),   # level 2 unsplit: 4 channels, 144 bricks
])
@pytest.mark.parametrize("mip", ["NEAREST", "LINEAR"])
def test_split_levels(ngt_ops, dims, out_dhw, C, n, views, levels, mip):  # noqa: F811
    rng = np.random.default_rng(4000 + dims[0] + 7 * C + 3 * views + levels)
    mip = mip if levels else "NONE"
    cams = cameras(dims, out_dhw, views, n, 3.0, 2.0, 4.0)
    inp = f32(rng.standard_normal((n,) + dims + (C,)))
    g = f32(rng.standard_normal((n, views) + out_dhw + (C,)))
    # NEAREST picks between levels at half steps, where fp32 and fp64 may
    # differ for a sample on one: a bias keeps this set of samples off them
    bias = 0.0 if mip == "LINEAR" else 0.0173
    exp = R.sample_grid_transform_grad(inp, g, *cams, LINEAR, BORDER, R.COORDINATE_MODE["TRANSFORM_LINDEPTH"], True,
                                       "exact", MP.MIPMODE[mip], levels, bias)
    got = host(ngt_ops.sample_grid_transform_grad(dev(inp), dev(g), *cams, coordinate_mode="TRANSFORM_LINDEPTH",
                                                  mipmapping=mip, num_mipmaps=levels, mip_bias=bias))
    assert rel(got, exp) < 1e-4
