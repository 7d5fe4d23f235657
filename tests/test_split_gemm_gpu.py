"""gemm_f32_sp: fp32 products on the bf16 units from operands cut into three
bf16 parts.  Every tile at its edges, both operand orders, operands off 16-byte
alignment, K remainders, split-K, the epilogue, and values that the cut cannot
hold (infinities, NaN, sums past the largest float, subnormals), against float64."""
import numpy as np
import pytest
import torch

import minitensor_amd as mt

pytestmark = pytest.mark.gpu
# (family, configuration, tile rows, tile columns)
TILES = [(mt.FAMILY_DL, 0, 64, 256), (mt.FAMILY_DL, 1, 128, 128), (mt.FAMILY_DL, 3, 256, 128),
         (mt.FAMILY_DL, 4, 128, 256), (mt.FAMILY_DL, 6, 128, 64),
         (mt.FAMILY_RS, 0, 256, 128), (mt.FAMILY_RS, 1, 128, 128), (mt.FAMILY_RS, 2, 64, 64)]


def operand(rng, rows, cols, k_major, off, dev, fill=None):
    """rows x cols, cols the contiguous index when k_major, `off` floats past an
    aligned address; `fill(a)` edits the values."""
    a = rng.standard_normal((rows, cols)).astype(np.float32)
    if fill:
        fill(a)
    src = a if k_major else np.ascontiguousarray(a.T)
    buf = torch.empty(src.size + 8, device=dev)
    buf[off:off + src.size] = torch.from_numpy(src.reshape(-1)).to(dev)
    t = buf[off:off + src.size].view(src.shape)
    return a, (t if k_major else t.t())


def check(got, a, b, extra, k):
    # each product rounded to 2^-24 and k sums: (k + 4)·2^-24·Σ|a||b| per element;
    # 2^-126: what is below the smallest normal float may be flushed
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want = a64 @ b64 + extra
    bound = (k + 4) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64) + np.abs(extra)) + 2.0 ** -126
    err = np.abs(got.double().cpu().numpy() - want)
    assert (err <= bound).all(), float((err / bound).max())
    # A product of the six that is lost somewhere (2.4e-6 of the result's 2-norm for
    # the smallest, from its definition on normal values) may hide below that bound:
    # 1.5 times the 6.4e-9 sqrt(k) measured for sums of k, and roundings of the result
    if want.size >= 1000 and k >= 16 and 1e-30 < np.abs(want).max() and np.abs(a).max() < 100:
        norm = float(np.linalg.norm(err) / np.linalg.norm(want))
        assert norm <= 3e-7 + 1.5 * 6.4e-9 * k ** 0.5, (norm, k, mt.last_config())


@pytest.mark.parametrize("fam,cfg,bm,bn", TILES)
@pytest.mark.parametrize("a_k,b_k", [(True, True), (True, False), (False, True), (False, False)])
def test_tile_edges(dev, fam, cfg, bm, bn, a_k, b_k):
    rng = np.random.default_rng(bm * 7 + bn + 2 * a_k + b_k)
    aligned = fam == mt.FAMILY_DL
    step = 4 if aligned else 1   # the direct family's extents: multiples of four
    sizes = [(step, step, step), (bm, bn, 16), (bm - step, bn + step, 32 + step),
             (bm + step, bn - step, 208 - step), (2 * bm + step, bn, 64), (bm, bn, 32)]
    for (m, n, k), splits in [(s, 1) for s in sizes] + [(sizes[3], 3)]:
        off = 0 if aligned else 1 + (m & 1)
        a, A = operand(rng, m, k, a_k, off, dev)
        b, B = operand(rng, n, k, b_k, off, dev)
        c = rng.standard_normal((m, n)).astype(np.float32)
        bias = rng.standard_normal(n).astype(np.float32)
        C = torch.from_numpy(c).to(dev)
        with mt.forced_config(fam, cfg, splits):
            mt.gemm(A, B.t(), out=C, bias=torch.from_numpy(bias).to(dev), bias_axis=mt.BIAS_COL,
                    beta=0.5)
        name = mt.last_config()
        assert name.startswith("dl " if aligned else "rs ") and name.endswith(f" cfg={cfg}"), name
        want = 0.5 * c.astype(np.float64) + bias
        check(C, a, np.ascontiguousarray(b.T), want, k)


@pytest.mark.parametrize("fam,cfg,bm,bn", TILES)
def test_values_outside_the_cut(dev, fam, cfg, bm, bn):
    rng = np.random.default_rng(cfg)
    m, n, k = 2 * bm, 2 * bn, 96
    top = np.finfo(np.float32).max

    def scaled(s):
        return lambda x: np.multiply(x, np.float32(s), out=x)

    for sa, sb in [(1e-38, 1e30), (1e-42, 1.0), (1e18, 1e18), (1e-20, 1e-20)]:
        a, A = operand(rng, m, k, True, 0, dev, scaled(sa))
        b, B = operand(rng, n, k, True, 0, dev, scaled(sb))
        with mt.forced_config(fam, cfg, 1):
            check(mt.gemm(A, B.t()), a, np.ascontiguousarray(b.T), 0.0, k)

    def odd(x):
        x[1, 3], x[5, 7], x[6, 0] = np.inf, np.nan, -np.inf
        x[9] = 0.0
        x[9, 2] = -top
        x[m - 1, k - 1] = top
    a, A = operand(rng, m, k, True, 0, dev, odd)
    b, B = operand(rng, n, k, True, 0, dev)
    with mt.forced_config(fam, cfg, 1):
        got = mt.gemm(A, B.t()).cpu().numpy()
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.T.astype(np.float64)
    assert np.isnan(got[5]).all()
    for r in (1, 6):
        assert (got[r] == want[r]).all()                    # ± infinity, by b's sign
    assert (got[9] == (a[9, 2] * b[:, 2].astype(np.float64)).astype(np.float32)).all()
    rest = [r for r in range(m - 1) if r not in (1, 5, 6, 9)]
    check(torch.from_numpy(got[rest]), a[rest], np.ascontiguousarray(b.T), 0.0, k)


@pytest.mark.parametrize("fam,cfg,bm,bn", TILES)
def test_worst_operands(dev, fam, cfg, bm, bn):
    """0x1.00ff8p+0 is cut into 1 + 2^-8 - 2^-17: the products left out come to 2^-24
    of each product, all of one sign, and grow with the sum."""
    v = float.fromhex("0x1.00ff8p+0")
    for k in (16, 256, 4096, 16384):
        with mt.forced_config(fam, cfg, 1):
            got = mt.gemm(torch.full((bm, k), v, device=dev), torch.full((k, bn), v, device=dev))
        # 2^-24 left out and 2^-24 of the last additions (h.h, all ones, sums exactly);
        # the small products are 2^-7 of the sum, which the unit rounds to 2^-23 and
        # not to nearest at each of 5 k/16 instructions
        bound = 2.0 ** -23 + 5 * k / 16 * 2.0 ** -30
        err = float((got.double() / (k * v * v) - 1).abs().max())
        print(f"[worst] {mt.last_config()} k={k} {err:.3g} of {bound:.3g}", flush=True)
        assert err <= bound, (k, err, bound)
