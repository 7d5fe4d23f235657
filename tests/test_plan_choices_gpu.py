"""Tiles and splits of calls that lost time when the larger ones moved to the bf16 units:
too few workgroups for the first loads or the store to run beside anything, short
ranges of K, both operands across rows.  (Times of the plan that each had taken,
and of the one it takes, stand beside the planner's prices.)"""
import pytest
import torch

import minitensor_amd as mt

pytestmark = pytest.mark.gpu


def conv(dev, n, c, h, co, k, stride, pad, part):
    x = torch.zeros(n, c, h, h, device=dev)
    w = torch.zeros(co, c, k, k, device=dev)
    if part == "fwd":
        mt.conv2d(x, w, None, stride, pad)
    else:
        ho = (h + 2 * pad - k) // stride + 1
        mt.conv2d_backward(x, w, torch.zeros(n, co, ho, ho, device=dev), stride, pad,
                           need_dx=part == "dx", need_dw=part == "dw", need_db=part == "dw")
    return mt.last_config()


def gemm(dev, m, n, k, ta=False, tb=False, beta=0.0):
    a = torch.zeros(k, m, device=dev).t() if ta else torch.zeros(m, k, device=dev)
    b = torch.zeros(n, k, device=dev).t() if tb else torch.zeros(k, n, device=dev)
    mt.gemm(a, b, out=torch.zeros(m, n, device=dev), beta=beta)
    return mt.last_config()


PLANS = [
    (lambda d: conv(d, 19, 112, 32, 144, 1, 1, 0, "fwd"), "64x64"),    # 64x256, one per CU
    (lambda d: conv(d, 15, 224, 32, 80, 1, 1, 0, "dx"), "64x64"),      # 128x128, one per CU
    (lambda d: gemm(d, 3904, 1120, 17, beta=0.5), "64x64"),            # 128x128, unaligned
    (lambda d: gemm(d, 2656, 2656, 144, ta=True), "256x128"),          # 128x128, both across
    (lambda d: gemm(d, 2832, 3904, 864, ta=True), "128x128"),          # ... long: stays
    (lambda d: gemm(d, 709, 2374, 396, tb=True), "64x64"),            # (128x64 would not hide)
    (lambda d: conv(d, 1, 96, 28, 416, 3, 1, 1, "fwd"), "64x64"),      # 64x112 in nine splits
    (lambda d: conv(d, 9, 8, 28, 80, 3, 1, 1, "dx"), "64x112"),        # ... stays where it won
    (lambda d: conv(d, 20, 80, 7, 240, 3, 1, 1, "dw"), "split=5"),     # 16, three per CU
    (lambda d: conv(d, 1, 32, 14, 112, 3, 1, 1, "dw"), "cfg=5"),       # the kernel without prefetch
    (lambda d: conv(d, 4, 16, 32, 48, 3, 1, 1, "dw"), "cfg=2"),        # ... with dY in NCHW stays
]


@pytest.mark.parametrize("case", range(len(PLANS)))
def test_tile(dev, case):
    call, tile = PLANS[case]
    got = call(dev) + " "
    assert f" {tile} " in got, got
