"""GPU parity of the LINEAR table adjoint, which adds a tile's corners in LDS
over their bounding box, against the FP64 oracle: tables off the tile's extents
and of one cell, tiles whose box fits, tiles of scattered positions whose box
does not, positions outside the grid and on cell centres, all boundaries,
channel counts and mip modes.

Tolerance: gradients 1e-4 of the largest value, as for the direct scatter.
"""
import numpy as np
import pytest
import torch

from oracle import BORDER, CLAMP, LINEAR, WRAP
from oracle import mips as MP
from oracle import resample as R

pytestmark = pytest.mark.gpu

BNAME = {BORDER: "BORDER", CLAMP: "CLAMP", WRAP: "WRAP"}
MNAME = {MP.MIP_NONE: "NONE", MP.MIP_NEAREST: "NEAREST", MP.MIP_LINEAR: "LINEAR"}


@pytest.fixture(scope="module")
def ngt_ops():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from ngt import ops, _lib
    _lib.load()
    return ops


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a, dtype=np.float32))).to("cuda:0")


def f32(a):
    return np.asarray(a, dtype=np.float32).astype(np.float64)


def rel(got, exp):
    return float(np.max(np.abs(got.detach().cpu().double().numpy() - exp))) / max(float(np.max(np.abs(exp))), 1e-30)


def table(rng, out_dhw, grid_dhw, views, kind, levels):
    """Absolute positions: 'warp' = the grid's extent stretched over the table
    with a jitter of one cell, reaching past the border; 'scatter' = anywhere
    within the grid and a little beyond; 'mixed' = warped for x < 16 (tiles
    whose box fits) and scattered after it.  Multiples of 1/64 plus 1/256: FP32
    and FP64 agree about the corners at every level."""
    idx = np.stack(np.meshgrid(*[np.arange(n) for n in out_dhw], indexing="ij"), -1)[..., ::-1]
    size = np.array(grid_dhw[::-1], dtype=np.float64)
    warp = (idx + 0.5) / np.array(out_dhw[::-1]) * (size + 3.0) - 1.5 + rng.uniform(-1, 1, (views,) + out_dhw + (3,))
    far = rng.uniform(-2.0, 1.0, (views,) + out_dhw + (3,)) + rng.uniform(0, 1, (views,) + out_dhw + (3,)) * (size + 2.0)
    pos = {"warp": warp, "scatter": far, "mixed": np.where(idx[..., :1] < 16, warp, far)}[kind]
    pos = np.round(pos * 64.0) / 64.0 + 1.0 / 256.0
    lod = rng.uniform(-0.5, levels + 0.5, (views,) + out_dhw + (1,))
    return f32(np.concatenate([pos, lod], -1))


@pytest.mark.parametrize("bound", [BORDER, CLAMP, WRAP])
@pytest.mark.parametrize("C,out_dhw,grid_dhw,kind,mip", [
    (1, (5, 9, 33), (7, 10, 21), "warp", MP.MIP_NONE),
    (1, (9, 17, 40), (20, 24, 28), "mixed", MP.MIP_NONE),
    (1, (6, 8, 16), (40, 30, 50), "scatter", MP.MIP_LINEAR),
    (2, (5, 7, 18), (9, 8, 20), "warp", MP.MIP_LINEAR),
    (2, (4, 9, 35), (20, 24, 28), "mixed", MP.MIP_NEAREST),
    (4, (5, 9, 17), (6, 9, 15), "warp", MP.MIP_NONE),
    (4, (5, 9, 17), (20, 24, 28), "mixed", MP.MIP_LINEAR),
    (1, (1, 1, 1), (3, 3, 3), "warp", MP.MIP_NONE),
    (4, (3, 2, 70), (1, 1, 40), "warp", MP.MIP_NONE),
])
def test_matches_oracle(ngt_ops, C, out_dhw, grid_dhw, kind, mip, bound):
    rng = np.random.default_rng(7000 + C + sum(out_dhw) + 31 * bound)
    levels = 0 if mip == MP.MIP_NONE else 2
    inp = f32(rng.standard_normal((2,) + grid_dhw + (C,)))
    lut = table(rng, out_dhw, grid_dhw, 2, kind, levels)
    g = f32(rng.standard_normal((2, 2) + out_dhw + (C,)))
    ei, el = R.sample_grid_lut_grad(inp, lut, g, LINEAR, bound, 0.5, True, False, False, "exact", mip, levels, 0.0)
    gi, gl = ngt_ops.sample_grid_lut_grad(dev(inp), dev(g), dev(lut), boundary=BNAME[bound], mipmapping=MNAME[mip],
                                          num_mipmaps=levels, cell_center_offset=0.5, relative_coords=False)
    assert rel(gi, ei) < 1e-4
    assert rel(gl, el) < 1e-4


@pytest.mark.parametrize("bound", [BORDER, CLAMP, WRAP])
def test_cell_centres_and_one_camera_per_entry(ngt_ops, bound):
    """Whole-number positions have one corner per axis: every sample's gradient
    goes to one cell, exactly."""
    rng = np.random.default_rng(7100 + bound)
    dims = (6, 9, 20)
    inp = f32(rng.integers(-3, 4, (2,) + dims + (1,)))
    lut = np.zeros((2,) + dims + (4,))
    lut[..., :3] = rng.integers(-2, 3, (2,) + dims + (3,))
    g = f32(rng.integers(-3, 4, (2, 1) + dims + (1,)))
    ei, _ = R.sample_grid_lut_grad(inp, lut, g, LINEAR, bound, 0.0, False, True, False, "exact")
    gi, _ = ngt_ops.sample_grid_lut_grad(dev(inp), dev(g), dev(lut), boundary=BNAME[bound], separate_camera_batch=False)
    assert np.array_equal(gi.cpu().numpy().astype(np.float64), ei)


def test_positions_that_are_no_number_do_not_spread(ngt_ops):
    """A NaN position is outside a BORDER grid; a NaN gradient reaches the
    corners of its own sample alone."""
    rng = np.random.default_rng(7200)
    inp = dev(rng.standard_normal((1, 6, 6, 20, 1)))
    lut = dev(rng.uniform(-0.4, 0.4, (1, 6, 6, 20, 4)))
    g = dev(rng.standard_normal((1, 1, 6, 6, 20, 1)))
    nan_lut, nan_g = lut.clone(), g.clone()
    nan_lut[0, 3, 3, 7, 0] = float("nan")
    nan_g[0, 0, 3, 3, 7, 0] = float("nan")
    zero_g = g.clone()
    zero_g[0, 0, 3, 3, 7, 0] = 0.0
    base, _ = ngt_ops.sample_grid_lut_grad(inp, zero_g, lut, separate_camera_batch=False)
    out, _ = ngt_ops.sample_grid_lut_grad(inp, g, nan_lut, separate_camera_batch=False)
    assert torch.allclose(out, base, atol=1e-5)
    hit, _ = ngt_ops.sample_grid_lut_grad(inp, nan_g, lut, separate_camera_batch=False)
    bad = torch.isnan(hit)
    assert 1 <= int(bad.sum()) <= 8 and torch.allclose(hit[~bad], base[~bad], atol=1e-5)
