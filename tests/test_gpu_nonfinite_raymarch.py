"""An image gradient that is no finite number shows in the ray adjoint's brick
gather: its sums are integers of a unit taken from a bound on the gradients, so
the bound has to carry the NaN or infinity of any sample and channel, whatever
follows it on the ray.  The scatter adjoint adds in float and serves as the
oracle: where it is not finite, the gather is not.
"""
import numpy as np
import pytest
import torch

from test_gpu_raymarch_gather import cameras, dev, ngt_ops  # noqa: F401  (the module's fixture)

pytestmark = pytest.mark.gpu

DIMS, OUT_DHW = (9, 8, 11), (14, 6, 10)


def check(ops, monkeypatch, C, blend, channel):
    rng = np.random.default_rng(40 + C + channel)
    cams = cameras(DIMS, OUT_DHW, 1, 20.0)
    x = dev(rng.uniform(0.01, 0.1, (1,) + DIMS + (C,)))
    out = ops.raymarch_grid_transform(x, *cams, OUT_DHW, blending_mode=blend)
    base = dev(rng.standard_normal(tuple(out.shape)))
    touched = 0
    # the pixels of a row and of a column: rays of odd and of even sample counts
    for row, col in [(2, c) for c in range(OUT_DHW[2])] + [(r, 4) for r in range(OUT_DHW[1])]:
        for bad in (float("nan"), float("inf")):
            g = base.clone()
            g[0, 0, row, col, channel] = bad
            grads = []
            for gather in (False, True):
                monkeypatch.setattr(ops, "use_gather_adjoint", gather)
                grads.append(ops.raymarch_grid_transform_grad(x, out, g, *cams, OUT_DHW, blending_mode=blend))
            expected = ~torch.isfinite(grads[0]).all(-1)
            touched += int(expected.any())
            assert not torch.isfinite(grads[1][expected]).all(-1).any(), (row, col, bad)
    assert touched > 20


@pytest.mark.parametrize("C,blend,channel",
                         [(1, "BEER_LAMBERT", 0), (2, "ADDITIVE", 0), (2, "ADDITIVE", 1), (2, "BEER_LAMBERT", 0)] +
                         [(4, b, c) for b in ("BEER_LAMBERT", "ALPHA_ADDITIVE") for c in range(4)])
def test_nonfinite_gradient_reaches_the_bound(ngt_ops, monkeypatch, C, blend, channel):  # noqa: F811
    check(ngt_ops, monkeypatch, C, blend, channel)


@pytest.mark.parametrize("blend", ["ADDITIVE", "ALPHA"])
@pytest.mark.parametrize("channel", range(4))
def test_nonfinite_colour_reaches_the_bound(ngt_ops, monkeypatch, blend, channel):  # noqa: F811
    """Blends whose last channel's gradient can stay finite beside a colour's that is not."""
    check(ngt_ops, monkeypatch, 4, blend, channel)
