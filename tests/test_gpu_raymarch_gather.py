"""GPU parity of the ray adjoint's brick gather against the scatter adjoint of
the same samples and against the FP64 oracle, where its dealing of samples to wavefronts changes: more samples per wavefront than
it marks at once (steps much shorter than a cell), image pixels closer than
cells, grids of one cell along an axis, extents off the bricks, more views than
one launch takes, rays that miss the grid, and every channel count.

Tolerance: gradients 1e-4 of the largest value, as for the other adjoints.
"""
import numpy as np
import pytest
import torch

from oracle import BORDER, LINEAR
from oracle import blend as B
from oracle import geometry as G
from oracle import raymarch as RM

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


def f32(a):
    return np.asarray(a, dtype=np.float32).astype(np.float64)


def rel(got, exp):
    return float(np.max(np.abs(got.detach().cpu().double().numpy() - exp))) / max(float(np.max(np.abs(exp))), 1e-30)


def cameras(dims, out_dhw, views, fov):
    M = G.grid_transform(dims, translation_=(0.0123, -0.0217, 0.0311), center=True, scale_=[1.0 / max(dims)] * 3)
    cams = G.look_at_ring_cameras(views, 3.0, fov, out_dhw[2] / out_dhw[1], 2.0, 4.0)
    return ([G.op_matrix(M).astype(np.float32)], [G.op_matrix(c[0]).astype(np.float32) for c in cams],
            [G.op_matrix(c[1]).astype(np.float32) for c in cams], [c[2].astype(np.float32) for c in cams])


@pytest.mark.parametrize("dims,out_dhw,C,views,fov,same_samples", [
    ((7, 9, 11), (400, 7, 9), 1, 2, 25.0, True),     # some 20 samples per cell: several marked parts
    ((7, 9, 11), (400, 7, 9), 4, 2, 25.0, True),
    ((6, 5, 7), (8, 48, 64), 1, 3, 25.0, True),      # many rays per cell
    ((6, 5, 7), (8, 48, 64), 2, 3, 25.0, True),
    # one cell along an axis; seen edge-on, a ray's first sample falls on either
    # side of the grid's face in FP32 and FP64 (the images differ too)
    ((1, 17, 33), (40, 9, 13), 1, 3, 25.0, False),
    ((17, 1, 1), (40, 9, 13), 4, 2, 25.0, False),
    ((18, 19, 17), (24, 11, 13), 4, 9, 60.0, True),  # two launches; rays beside the grid
    ((18, 19, 17), (24, 11, 13), 2, 3, 60.0, True),
])
def test_matches_scatter_and_oracle(ngt_ops, monkeypatch, dims, out_dhw, C, views, fov, same_samples):
    rng = np.random.default_rng(8000 + C + sum(dims) + views)
    Ms, Vs, Ps, Fs = cameras(dims, out_dhw, views, fov)
    x = f32(rng.uniform(0.0, 0.5, (1,) + dims + (C,)) * 20.0 / out_dhw[0])
    exp = RM.raymarch_grid_transform(x, Ms, Vs, Ps, Fs, out_dhw, LINEAR, BORDER, B.BEER_LAMBERT)
    g = f32(rng.standard_normal(exp.shape))
    eg = RM.raymarch_grid_transform_grad(x, exp, g, Ms, Vs, Ps, Fs, out_dhw, LINEAR, BORDER, B.BEER_LAMBERT)
    got = ngt_ops.raymarch_grid_transform_grad(dev(x), dev(exp), dev(g), Ms, Vs, Ps, Fs, out_dhw)
    monkeypatch.setattr(ngt_ops, "use_gather_adjoint", False)
    scatter = ngt_ops.raymarch_grid_transform_grad(dev(x), dev(exp), dev(g), Ms, Vs, Ps, Fs, out_dhw)
    assert rel(got, scatter.cpu().double().numpy()) < 1e-4
    if same_samples:
        assert rel(got, eg) < 1e-4


@pytest.mark.parametrize("dims,C", [((9, 100, 121), 1), ((72, 100, 100), 1), ((101, 113, 120), 1), ((101, 113, 120), 2)])
def test_brick_shapes_match_scatter(ngt_ops, monkeypatch, dims, C):
    """Grids that take bricks of 8^3, 16 x 8 x 8 and 16^3 cells, off their extents."""
    out_dhw = (48, 21, 30)
    rng = np.random.default_rng(8100 + sum(dims))
    Ms, Vs, Ps, Fs = cameras(dims, out_dhw, 3, 30.0)
    x = dev(rng.uniform(0.0, 0.5, (1,) + dims + (C,)))
    out = ngt_ops.raymarch_grid_transform(x, Ms, Vs, Ps, Fs, out_dhw)
    g = dev(rng.standard_normal(tuple(out.shape)))
    got = ngt_ops.raymarch_grid_transform_grad(x, out, g, Ms, Vs, Ps, Fs, out_dhw)
    monkeypatch.setattr(ngt_ops, "use_gather_adjoint", False)
    scatter = ngt_ops.raymarch_grid_transform_grad(x, out, g, Ms, Vs, Ps, Fs, out_dhw)
    assert rel(got, scatter.cpu().double().numpy()) < 1e-4


def test_thresholds_of_a_one_cell_grid():
    """q < the largest valid position (n - 0.5; for one cell the float below 0.5)
    is q + 0.5f < n in float, at the last floats below."""
    for n in (1, 2, 3, 4, 7, 8, 127, 128, 129, 4096):
        end = np.float32(0.5) - np.float32(2.0) ** -25 if n == 1 else np.float32(n) - np.float32(0.5)
        q = np.float32(n) - np.float32(0.5)
        for _ in range(12):
            assert (q < end) == (np.float32(q + np.float32(0.5)) < np.float32(n)), (n, q)
            q = np.nextafter(q, np.float32(-1.0))
