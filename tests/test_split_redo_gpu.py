"""Tiles of gemm_f32_sp whose sums are not finite are taken again with fp32 MFMAs:
every operand form, with K splits, batches and the fused row sums, has infinities
and NaNs where float64 has them and the other values as close as ever."""
import numpy as np
import pytest
import torch

import minitensor_amd as mt
import oracle

pytestmark = pytest.mark.gpu
DL = mt.FAMILY_DL


def same(got, want, k, scale, what):
    got = got.double().cpu().numpy()
    want = want.numpy() if isinstance(want, torch.Tensor) else want
    assert np.array_equal(np.isnan(got), np.isnan(want)), (what, mt.last_config())
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(got), inf) and (got[inf] == want[inf]).all(), what
    ok = np.isfinite(want)
    # k products of at most `scale`, each rounded to 2^-24 and summed in chunks
    err = np.abs(got[ok] - want[ok]).max()
    assert err <= max(k, 4) * 2.0 ** -24 * scale, (what, err)
    assert not ok.all() and ok.any(), what


def finite_max(a):
    return float(np.abs(a[np.isfinite(a)]).max())


def gpu(a, dev, across=False):
    if across:
        return torch.from_numpy(np.ascontiguousarray(a.swapaxes(-1, -2))).to(dev).transpose(-1, -2)
    return torch.from_numpy(a).to(dev)


@pytest.mark.parametrize("fam,cfg", [(DL, 0), (DL, 1), (DL, 3), (DL, 4), (DL, 6), (mt.FAMILY_RS, 0),
                                     (mt.FAMILY_RS, 1), (mt.FAMILY_RS, 2)])
@pytest.mark.parametrize("a_across,b_across", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("batch,splits", [(1, 3), (3, 1), (2, 2)])
def test_products(dev, fam, cfg, a_across, b_across, batch, splits):
    off = 0 if fam == DL else 1          # the other family: rows off 16-byte alignment
    m, n, k = 300 + off, 260 + off, 148 + off
    a, b = oracle.normal((batch, m, k), 31), oracle.normal((batch, k, n), 32)
    a[0, 1, 3], a[0, 5, 70], a[-1, m - 1, k - 1] = np.inf, np.nan, -np.inf
    b[-1, 100, n - 1] = np.inf
    A, B = gpu(a, dev, a_across), gpu(b, dev, not b_across)
    if batch == 1:
        A, B = A[0], B[0]
    with mt.forced_config(fam, cfg, splits):
        got = mt.gemm(A, B)
        name = mt.last_config()
    assert f" split={splits} " in name and name.endswith(f" cfg={cfg}"), name
    want = (torch.from_numpy(a).double() @ torch.from_numpy(b).double()).numpy()
    same(got if batch > 1 else got[None], want, k, finite_max(a) * finite_max(b), name)


# n, c, h, c_out, k, stride, pad, operand: channels-last; the NCHW view without
# and (1x1: no halo patches) with the gather of this kernel
@pytest.mark.parametrize("layer,cfgs", [((3, 32, 17, 70, 3, 1, 1, "im2col "), (0, 1, 3, 7)),
                                        ((3, 20, 17, 70, 1, 1, 1, "im2col_nchw "), (0, 1, 3))])
@pytest.mark.parametrize("splits", [1, 2])
def test_forward(dev, layer, cfgs, splits):
    n, c, h, co, k, s, p, form = layer
    x, w = oracle.normal((n, c, h, h), 33), oracle.normal((co, c, k, k), 34)
    x[0, 3, 5, 5], x[1, 9, 0, 16], x[2, c - 1, 16, 16] = np.inf, np.nan, -np.inf
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(),
                                      stride=s, padding=p)
    if p >= k:   # (padded pixels of a 1x1: nothing but zeros)
        assert (want[:, :, 0] == 0).all()
    for cfg in cfgs:
        with mt.forced_config(DL, cfg, splits):
            y = mt.conv2d(gpu(x, dev), gpu(w, dev), None, s, p)
            name = mt.last_config()
        assert f"b={form}" in name and name.endswith(f" cfg={cfg}"), name
        same(y, want, c * k * k, finite_max(x) * finite_max(w), name)


# The padded stem: a tile of 128 x 128, and the 64 x 112 one of larger layers (12
# images of 2601 pixels end in the middle of a tile)
@pytest.mark.parametrize("layer,tile", [((2, 3, 37, 64), "128x128"), ((12, 3, 101, 64), "64x112")])
def test_stem_forward(dev, layer, tile):
    n, c, h, co = layer
    x, w = oracle.normal((n, c, h, h), 35), oracle.normal((co, c, 7, 7), 36)
    X, W = gpu(x, dev), gpu(w, dev)
    y = mt.conv2d(X, W, None, 2, 3)
    name = mt.last_config()
    assert f" {tile} " in name and "im2col_nchw_c4" in name, name
    scale = float(np.abs(x).max() * np.abs(w).max())
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(),
                                      stride=2, padding=3)
    assert float((y.double().cpu() - want).abs().max()) <= c * 49 * 2.0 ** -24 * scale
    x[0, 1, 5, 5], x[n - 1, 2, h - 1, h - 1] = np.nan, np.inf
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(),
                                      stride=2, padding=3)
    same(mt.conv2d(gpu(x, dev), W, None, 2, 3), want, c * 49, scale, name)


def weight_gradient64(x, dy, k, s, p):
    co, c = dy.shape[1], x.shape[1]
    w = torch.zeros(co, c, k, k, dtype=torch.float64, requires_grad=True)
    y = torch.nn.functional.conv2d(torch.from_numpy(x).double(), w, stride=s, padding=p)
    return torch.autograd.grad(y, w, torch.from_numpy(dy).double())[0]


# dY read in NCHW (whole groups of four pixels and chunks), and copied
@pytest.mark.parametrize("layer,form", [((4, 32, 16, 70), "a=kv_nchw"), ((4, 32, 17, 70), "a=kv ")])
@pytest.mark.parametrize("cfg,splits", [(0, 1), (0, 3), (0, 40), (3, 1), (3, 3)])
def test_weight_gradient(dev, layer, form, cfg, splits):
    n, c, h, co = layer
    x, dy = oracle.normal((n, c, h, h), 37), oracle.normal((n, co, h, h), 38)
    x[0, 3, 5, 5], x[1, 9, 2, 2] = np.inf, np.nan
    dy[2, 11, 4, 4] = -np.inf
    with mt.forced_config(DL, cfg, splits):
        dw, db = mt.conv2d_backward(gpu(x, dev), torch.zeros(co, c, 3, 3, device=dev), gpu(dy, dev),
                                    1, 1, need_dx=False)[1:]
        name = mt.last_config()
    assert form in name and "b=im2colT" in name and name.endswith(f" cfg={cfg}"), name
    # configuration 0 with splits hands the row sums of dY to the reduction
    assert (" rows " in name) == (cfg == 0 and splits > 1), name
    k = n * h * h
    same(dw, weight_gradient64(x, dy, 3, 1, 1), k, finite_max(x) * finite_max(dy), name)
    same(db, dy.astype(np.float64).sum((0, 2, 3)), k, finite_max(dy), name)


# db out of the dW products: two operands across (Linear), two along k summed over
# the images (1x1 layers)
@pytest.mark.parametrize("cfg", [0, 1, 3, 4, 6])
def test_row_sums(dev, cfg):
    rows, fin, fout = 200, 260, 136
    x, dy = oracle.normal((rows, fin), 39), oracle.normal((rows, fout), 40)
    x[3, 5], dy[100, 7], dy[101, 8] = np.nan, np.inf, np.nan
    with mt.forced_config(DL, cfg, 1):
        dw, db = mt.linear_backward(gpu(dy, dev), gpu(x, dev), torch.zeros(fout, fin, device=dev),
                                    need_dx=False)[1:]
        name = mt.last_config()
    assert " rows " in name and name.endswith(f" cfg={cfg}"), name
    y64, x64 = dy.astype(np.float64), x.astype(np.float64)
    same(dw, y64.T @ x64, rows, finite_max(x) * finite_max(dy), name)
    same(db, y64.sum(0), rows, finite_max(dy), name)

    n, c, h, co = 3, 260, 12, 136
    x, dy = oracle.normal((n, c, h, h), 41), oracle.normal((n, co, h, h), 42)
    x[0, 3, 5, 5], dy[1, 7, 2, 2], dy[2, 8, 4, 4] = np.nan, np.inf, np.nan
    with mt.forced_config(DL, cfg, 1):
        dw, db = mt.conv2d_backward(gpu(x, dev), torch.zeros(co, c, 1, 1, device=dev), gpu(dy, dev),
                                    1, 0, need_dx=False)[1:]
        name = mt.last_config()
    assert "batch-summed rows" in name and f" cfg={cfg} " in name, name
    same(dw, weight_gradient64(x, dy, 1, 1, 0), n * h * h, finite_max(x) * finite_max(dy), name)
    same(db, dy.astype(np.float64).sum((0, 2, 3)), n * h * h, finite_max(dy), name)
