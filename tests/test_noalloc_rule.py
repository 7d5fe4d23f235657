"""Which products mt_gemm_noalloc_f32 takes is a rule on their sizes that does
not move with the planner's prices: sizes on both sides of the limit."""
import ctypes

import pytest

import minitensor_amd as mt

REFUSED = [(2505, 194, 2811, 9), (198, 11659, 1612, 1), (331, 4441, 5789, 1), (197, 9583, 2310, 1),
           (444, 1544, 6492, 1), (12083, 97, 3030, 1), (3802, 546, 11852, 1), (70, 9819, 5167, 1)]
TAKEN = [(1016, 1356, 1094, 1), (192, 2817, 10420, 1), (816, 2962, 6688, 1), (753, 235, 15699, 2),
         (12955, 116, 1603, 1), (3759, 61, 3135, 5), (960, 1107, 11159, 1), (7721, 29, 1922, 17),
         (3265, 4454, 4324, 1), (4096, 4096, 4096, 1), (1, 1, 1, 1)]


def mats(size):
    m, n, k, batch = size
    return [ctypes.byref(mt.MatF32(4096, 0, r, c, c, 1, batch, r * c))   # (never read)
            for r, c in ((m, k), (k, n), (m, n))]


@pytest.mark.parametrize("size", REFUSED)
def test_refused_before_any_launch(size):
    assert mt.lib().mt_gemm_noalloc_f32(*mats(size), None, None) == mt.MT_ERR_SCRATCH_LIMIT


@pytest.mark.parametrize("size", TAKEN)
def test_taken_sizes_plan_within_the_scratch(size):
    # (a query only: a taken call would launch)
    assert mt.lib().mt_gemm_workspace_f32(*mats(size)) <= mt.NOALLOC_SCRATCH_BYTES
