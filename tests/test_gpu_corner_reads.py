"""GPU parity of the 8-corner reads against the FP64 oracle where their addresses
are formed in different ways: wavefronts whose samples all lie between cells,
wavefronts that hold samples at, across and far beyond the grid's ends, samples
on cell centres, grids of one cell along an axis; every boundary and channel count.

Tolerance: positions and weights are exact, and each of the three lerps rounds a
difference and a sum: 3 * 2 * 2^-24 of twice the largest value, 7.2e-7; 1e-6.
"""
import numpy as np
import pytest

from oracle import BORDER, CLAMP, LINEAR, WRAP
from oracle import resample as R
from test_gpu_lut_tiles import BNAME, dev, f32, ngt_ops, rel  # noqa: F401  (the module's fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bound", [BORDER, CLAMP, WRAP])
@pytest.mark.parametrize("C", [1, 2, 4])
@pytest.mark.parametrize("dims", [(6, 7, 70), (3, 2, 5), (1, 9, 66), (5, 1, 2), (4, 6, 1)])
def test_linear_reads(ngt_ops, dims, C, bound):  # noqa: F811
    rng = np.random.default_rng(60 + 5 * C + sum(dims) + bound)
    out_dhw = (3, 8, 192)  # along x: a wavefront between cells, one across the ends, one anywhere
    size = np.array(dims[::-1], dtype=np.float64)
    u = rng.uniform(0.0, 1.0, (1,) + out_dhw + (3,))
    pos = np.concatenate([u[..., :64, :] * np.maximum(size - 1.0, 0.0),
                          np.where(u[..., 64:128, :] < 0.5, u[..., 64:128, :] * 4.0 - 1.5, size + u[..., 64:128, :] * 4.0 - 3.5),
                          (u[..., 128:, :] - 0.5) * 6.0 * size], axis=3)
    pos = np.round(pos * 64.0) / 64.0
    pos[..., :64, :] += 1.0 / 128.0          # never on a cell's centre
    pos[:, :, :, 64::3] = np.round(pos[:, :, :, 64::3])  # on one
    lut = f32(np.concatenate([pos, np.zeros_like(pos[..., :1])], -1))
    inp = f32(rng.standard_normal((1,) + dims + (C,)))
    exp = R.sample_grid_lut(inp, lut, LINEAR, bound, relative=False)
    got = ngt_ops.sample_grid_lut(dev(inp), dev(lut), boundary=BNAME[bound], relative_coords=False)
    assert rel(got, exp) < 1e-6
