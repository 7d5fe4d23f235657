"""Tiles and splits of calls that lost time when the larger ones moved to the bf16 units:
too few workgroups for the first loads or the store to run beside anything, short
ranges of K, both operands across rows, rows off 16-byte alignment, layers over an
NCHW view (halo patches on the fp32 units, or gathers on the bf16 ones).  (Times of the plan that each had taken,
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
    (lambda d: gemm(d, 432, 24304, 9), "64x64"),                       # 128x128
    (lambda d: gemm(d, 3710, 2591, 64), "64x64"),                      # 128x128
    (lambda d: gemm(d, 2407, 2861, 1500), "256x128"),                  # ... long: stays
    (lambda d: gemm(d, 4096, 4096, 48), "128x128"),                    # 64x64, 4096 of them
    (lambda d: gemm(d, 2048, 2048, 48), "64x64"),                      # ... fewer: stays
    (lambda d: conv(d, 10, 100, 7, 444, 5, 1, 2, "fwd"), "64x64"),     # 128x128 in 16 splits
    (lambda d: conv(d, 7, 24, 56, 120, 3, 1, 1, "fwd"), "64x64"),      # 128x128, one per CU
    (lambda d: conv(d, 32, 132, 14, 260, 3, 1, 1, "dx"), "b=im2col_halo"),
]


@pytest.mark.parametrize("case", range(len(PLANS)))
def test_tile(dev, case):
    call, tile = PLANS[case]
    got = call(dev) + " "
    assert f" {tile} " in got, got


# fwd and dX over an NCHW view, by stride phase, with the weights' copy, padded to four
# channels, channels-last
@pytest.mark.parametrize("layer", [(10, 100, 7, 444, 5, 1, 2), (4, 104, 14, 28, 3, 1, 1),
                                   (2, 24, 28, 36, 3, 2, 1), (3, 44, 13, 60, 5, 1, 2),
                                   (2, 3, 37, 64, 7, 2, 3), (1, 64, 9, 48, 3, 1, 1)])
def test_queried_workspace_holds_the_plan(dev, layer):
    """The plan with the workspace that the query asks for is the one with any more."""
    n, c, h, co, k, s, p = layer
    x = torch.zeros(n, c, h, h, device=dev)
    w = torch.zeros(co, c, k, k, device=dev)
    big = mt.workspace(1 << 28, dev)
    dy = torch.zeros_like(mt.conv2d(x, w, None, s, p))
    names = [mt.last_config()]
    mt.conv2d(x, w, None, s, p, ws=big)
    assert mt.last_config() == names[0]
    for need in ((True, False), (False, True)):
        got = []
        for ws in (None, big):
            mt.conv2d_backward(x, w, dy, s, p, need_dx=need[0], need_dw=need[1], need_db=need[1],
                               ws=ws)
            got.append(mt.last_config())
        assert got[0] == got[1], got
        names.append(got[0])
    print(names, flush=True)
