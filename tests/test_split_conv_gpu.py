"""The RGB stem's kernels and the weight gradient of gemm_f32_sp: four channels
per 16-byte load from a padded channels-last copy, the gather of a 64x256 dW
tile with the row sums that become db, and the reduction of many slabs, where
their tiles end, against float64."""
import numpy as np
import pytest
import torch

import minitensor_amd as mt
import oracle

pytestmark = pytest.mark.gpu

# n, c, h, w, c_out, k, stride, pad: a partial pixel tile and a partial channel
# tile; one image smaller than a tile; c_out past one tile; c = 1 and 2 stay off
# the padded path.  (All of them 128 x 128 tiles; 64 x 112 ones: test_split_redo_gpu.py.)
STEMS = [(2, 3, 37, 41, 64, 7, 2, 3), (1, 3, 9, 9, 5, 5, 1, 2), (3, 3, 30, 22, 130, 7, 2, 0),
         (2, 7, 12, 17, 33, 5, 1, 2), (2, 2, 21, 21, 20, 7, 1, 3), (32, 3, 19, 19, 64, 7, 2, 3)]
# ... for dW, on the plan's own tiles and on 64x256 ones: several tiles of columns,
# K not a multiple of 16, rows past one tile
LAYERS = [(8, 64, 28, 28, 64, 3, 1, 1), (40, 20, 28, 28, 64, 3, 1, 1), (5, 16, 27, 29, 70, 3, 1, 1),
          (32, 4, 56, 56, 48, 5, 2, 2)]


def conv64(x, w, s, p):
    return torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(),
                                      stride=s, padding=p)


def close(got, want, k, scale, what):
    # k products of magnitude <= scale, each rounded to 2^-24 and summed in
    # chunks: k·2^-24·scale bounds the sum of all roundings for k >= 4
    diff = got.double().cpu() - want
    err = float(diff.abs().max())
    assert err <= max(k, 4) * 2.0 ** -24 * scale, (what, err, k, scale)
    return float(diff.norm() / want.norm())


def lost_none(norm, k, what):
    # a lost product of the six shows as 2.4e-6 of the 2-norm or more (normal
    # values); 1.5 times the 6.4e-9 sqrt(k) measured for sums of k
    assert norm <= 3e-7 + 1.5 * 6.4e-9 * k ** 0.5, (what, norm, k, mt.last_config())


@pytest.mark.parametrize("shape", STEMS)
def test_stem_forward(dev, shape):
    n, c, h, w, co, k, s, p = shape
    x, wt = oracle.normal((n, c, h, w), 1), oracle.normal((co, c, k, k), 2)
    b = oracle.normal((co,), 3)
    y = mt.conv2d(torch.from_numpy(x).to(dev), torch.from_numpy(wt).to(dev),
                  torch.from_numpy(b).to(dev), stride=s, padding=p)
    assert ("im2col_nchw_c4" in mt.last_config()) == (c in (3, 7)), mt.last_config()
    want = conv64(x, wt, s, p) + torch.from_numpy(b).double()[None, :, None, None]
    norm = close(y, want, c * k * k + 1, float(np.abs(x).max() * np.abs(wt).max()), shape)
    if c in (3, 7):
        lost_none(norm, c * k * k, shape)


@pytest.mark.parametrize("shape", STEMS + LAYERS)
@pytest.mark.parametrize("splits", [0, 1, 3, 40])   # (from 32 on the reduction goes in slices)
def test_weight_gradient(dev, shape, splits):
    n, c, h, w, co, k, s, p = shape
    x = oracle.normal((n, c, h, w), 4)
    ho, wo = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
    dy = oracle.normal((n, co, ho, wo), 5)
    X, dY = torch.from_numpy(x).to(dev), torch.from_numpy(dy).to(dev)
    W = torch.zeros(co, c, k, k, device=dev)

    def run():
        return mt.conv2d_backward(X, W, dY, stride=s, padding=p, need_dx=False)[1:]

    if splits:
        with mt.forced_config(mt.FAMILY_DL, 0, splits):
            dw, db = run()
        if "b=im2colT" in mt.last_config():   # (c = 1, 2: a product of columns)
            assert " 64x256 " in mt.last_config(), mt.last_config()
    else:
        dw, db = run()
    x64 = torch.from_numpy(x).double()
    w64 = torch.zeros(co, c, k, k, dtype=torch.float64, requires_grad=True)
    y = torch.nn.functional.conv2d(x64, w64, stride=s, padding=p)
    (want,) = torch.autograd.grad(y, w64, torch.from_numpy(dy).double())
    m = n * ho * wo
    norm = close(dw, want, m, float(np.abs(x).max() * np.abs(dy).max()), shape)
    if splits:
        lost_none(norm, m, shape)
    close(db, torch.from_numpy(dy).double().sum((0, 2, 3)), m, float(np.abs(dy).max()), shape)


def test_weight_gradient_non_finite(dev):
    # the same elements are non-finite as in a plain product, whatever the plan
    # (tiles taken again on the fp32 units: test_split_redo_gpu.py)
    n, c, h, co = 8, 64, 28, 64
    x, dy = oracle.normal((n, c, h, h), 6), oracle.normal((n, co, h, h), 7)
    x[0, 3, 5, 5] = np.inf
    x[1, 9, 2, 2] = np.nan
    dy[2, 11, 4, 4] = -np.finfo(np.float32).max
    X, dY = torch.from_numpy(x).to(dev), torch.from_numpy(dy).to(dev)
    dw, db = mt.conv2d_backward(X, torch.zeros(co, c, 3, 3, device=dev), dY, stride=1, padding=1,
                                need_dx=False)[1:]
    dw = dw.cpu()
    assert torch.isnan(dw[:, 9]).all()
    assert not torch.isfinite(dw[:, 3]).any()
    clean = [i for i in range(c) if i not in (3, 9)]
    rows = [i for i in range(co) if i != 11]
    assert torch.isfinite(dw[rows][:, clean]).all()
    assert torch.isfinite(db[rows].cpu()).all()
