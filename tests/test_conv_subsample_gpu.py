"""Strided 1x1 layers: the pixels that they read copied out (two 16-byte loads
for four outputs, single floats where rows are odd, unaligned or short), the
product per image on them, and dX interleaved, against float64."""
import numpy as np
import pytest
import torch

import minitensor_amd as mt
import oracle

pytestmark = pytest.mark.gpu
# n, c, h, w, c_out, stride, view: even and odd widths (2*w_out past the row or
# not), w_out not a multiple of four, strides 3 and 4, one column, the first pixels
# off 16-byte alignment, rows and channels of a larger tensor
LAYERS = [(2, 16, 8, 8, 24, 2, ""), (3, 32, 15, 15, 16, 2, ""), (2, 16, 7, 23, 20, 2, ""),
          (1, 16, 4, 31, 8, 2, ""), (2, 48, 12, 12, 40, 3, ""), (2, 16, 13, 16, 64, 4, ""),
          (4, 64, 56, 56, 130, 2, ""), (2, 16, 8, 8, 24, 2, "off"), (2, 16, 8, 16, 24, 2, "crop"),
          (2, 16, 8, 8, 24, 2, "channels"), (2, 16, 8, 8, 24, 2, "nhwc"), (5, 16, 8, 1, 8, 2, "")]


def view_of(x, kind, dev):
    n, c, h, w = x.shape
    t = torch.from_numpy(x).to(dev)
    if kind == "off":
        buf = torch.zeros(x.size + 1, device=dev)
        v = buf[1:].view(x.shape)
    elif kind == "crop":
        v = torch.zeros(n, c, h + 2, w + 5, device=dev)[:, :, 1:h + 1, 2:w + 2]
    elif kind == "channels":
        v = torch.zeros(n, 2 * c, h, w, device=dev)[:, 1:2 * c:2]
    elif kind == "nhwc":
        v = torch.zeros(n, h, w, c, device=dev).permute(0, 3, 1, 2)
    else:
        return t
    v.copy_(t)
    return v


@pytest.mark.parametrize("layer", LAYERS)
def test_strided_pointwise(dev, layer):
    n, c, h, w, co, s, kind = layer
    x, wt = oracle.normal((n, c, h, w), 11), oracle.normal((co, c, 1, 1), 12)
    b = oracle.normal((co,), 13)
    X, W = view_of(x, kind, dev), torch.from_numpy(wt).to(dev)
    y = mt.conv2d(X, W, torch.from_numpy(b).to(dev), stride=s)
    x64 = torch.from_numpy(x).double().requires_grad_()
    w64 = torch.from_numpy(wt).double().requires_grad_()
    want = torch.nn.functional.conv2d(x64, w64, stride=s)
    scale = float(np.abs(x).max() * np.abs(wt).max())
    # (k + 4) roundings of 2^-24 of products of at most `scale`, and the bias
    got = y.double().cpu() - torch.from_numpy(b).double()[None, :, None, None]
    assert float((got - want.detach()).abs().max()) <= (c + 8) * 2.0 ** -24 * max(scale, 1.0)
    dy = oracle.normal(tuple(want.shape), 14)
    dx, dw, db = mt.conv2d_backward(X, W, torch.from_numpy(dy).to(dev), stride=s)
    gx, gw = torch.autograd.grad(want, (x64, w64), torch.from_numpy(dy).double())
    a = float(np.abs(dy).max())
    for got, ref, k, m in [(dx, gx, co, np.abs(wt).max()), (dw, gw, dy[:, 0].size, np.abs(x).max()),
                           (db, torch.from_numpy(dy).double().sum((0, 2, 3)), dy[:, 0].size, 1.0)]:
        assert float((got.double().cpu() - ref).abs().max()) <= (k + 4) * 2.0 ** -24 * a * float(m)
