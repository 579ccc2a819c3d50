"""GPU parity of the fused tables of a MAC velocity's self-advection with the
composed reads (resampling by a table per component, concatenation, product):
extents of one cell, odd extents and off the launch's blocks, several
instances, strided inputs, both boundaries, and gradients of some components
only; and which grids keep the composed reads.

Tolerance: values are the same reads, equal bit for bit; gradients sum up to 9
terms in another order, 2e-6 of the largest value.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ngt():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from ngt import _lib, data_structures, ops, renderer
    _lib.load()

    class Modules:
        pass

    m = Modules()
    m.ops, m.VelocityGrid, m.Renderer = ops, data_structures.VelocityGrid, renderer.Renderer
    return m


def faces(dhw, n, seed):
    g = torch.Generator().manual_seed(seed)
    d, h, w = dhw
    return [torch.randn(s, generator=g).cuda() for s in ((n, d, h, w + 1, 1), (n, d, h + 1, w, 1), (n, d + 1, h, w, 1))]


def grid(ngt, dhw, comps, boundary="BORDER", filter_mode="LINEAR"):
    r = ngt.Renderer(filter_mode=filter_mode, boundary_mode=boundary, mipmapping="NONE")
    return ngt.VelocityGrid(list(dhw), x=comps[0], y=comps[1], z=comps[2], warp_renderer=r)


def composed(v, scale):
    return [v._sampled_to_component_shape(c) * scale for c in "XYZ"]


@pytest.mark.parametrize("boundary", ["BORDER", "CLAMP"])
@pytest.mark.parametrize("dhw,n", [((1, 1, 1), 1), ((1, 4, 7), 1), ((5, 1, 3), 2), ((7, 9, 1), 1), ((9, 17, 63), 1),
                                   ((3, 5, 64), 3), ((8, 16, 65), 1)])
def test_matches_composed(ngt, dhw, n, boundary):
    comps = [c.requires_grad_() for c in faces(dhw, n, 3)]
    v = grid(ngt, dhw, comps, boundary)
    fused, exp = v._fused_component_luts(-0.7), composed(v, -0.7)
    for a, b in zip(fused, exp):
        assert a.shape == b.shape and torch.equal(a, b)
    up = [torch.randn_like(a) for a in fused]
    got = torch.autograd.grad(fused, comps, up)
    want = torch.autograd.grad(exp, comps, up)
    for a, b in zip(got, want):
        assert a.shape == b.shape and float((a - b).abs().max()) <= 2e-6 * float(b.abs().max())


def test_strided_components_and_partial_gradients(ngt):
    dhw = (6, 7, 10)
    x, y, z = faces(dhw, 1, 5)
    y = y.transpose(1, 3).contiguous().transpose(1, 3).requires_grad_()  # other strides
    v = grid(ngt, dhw, (x, y, z))
    fused, exp = v._fused_component_luts(2.0), composed(v, 2.0)
    assert all(torch.equal(a, b) for a, b in zip(fused, exp))
    up = torch.randn_like(fused[0]).transpose(1, 2).contiguous().transpose(1, 2)
    got, = torch.autograd.grad(fused[0], [y], up)  # one table's gradient alone
    want, = torch.autograd.grad(exp[0], [y], up)
    assert float((got - want).abs().max()) <= 2e-6 * float(want.abs().max())


def test_composed_reads_are_kept(ngt):
    dhw = (4, 5, 6)
    comps = faces(dhw, 1, 7)
    assert grid(ngt, dhw, comps)._fused_component_luts(-1.0) is not None
    assert grid(ngt, dhw, comps, "WRAP")._fused_component_luts(-1.0) is None
    assert grid(ngt, dhw, comps, filter_mode="NEAREST")._fused_component_luts(-1.0) is None
    assert grid(ngt, dhw, comps)._fused_component_luts(torch.tensor(-1.0)) is None
    assert grid(ngt, (4, 5, 7), comps)._fused_component_luts(-1.0) is None
    with ngt.ops.semantics("reference"):
        assert grid(ngt, dhw, comps)._fused_component_luts(-1.0) is None
    v = grid(ngt, dhw, comps, "WRAP")  # and still warp
    assert [t.shape for t in v.warped(order=2, clamp="MC_SMOOTH")] == [c.shape for c in comps]


@pytest.mark.parametrize("boundary", ["BORDER", "CLAMP"])
def test_warped_by_another_velocity(ngt, boundary, monkeypatch):
    dhw = (6, 9, 11)
    a, b = grid(ngt, dhw, faces(dhw, 1, 11), boundary), grid(ngt, dhw, faces(dhw, 1, 13), boundary)
    got = a.warped(b, order=2, dt=0.5, clamp="MC_SMOOTH")
    monkeypatch.setattr(ngt.VelocityGrid, "_fused_component_luts", lambda self, scale: None)
    want = a.warped(b, order=2, dt=0.5, clamp="MC_SMOOTH")
    assert all(torch.equal(p, q) for p, q in zip(got, want))


@pytest.mark.parametrize("boundary,shape,code", [("WRAP", (3, 4, 5), NotImplementedError),
                                                 ("BORDER", (3, 4, 6), ValueError)])
def test_refusals(ngt, boundary, shape, code):
    x, y, z = faces((3, 4, 5), 1, 1)
    with pytest.raises(code):
        ngt.ops.mac_component_luts(faces(shape, 1, 2)[0], y, z, 1.0, boundary)
