"""Workspace queries of many shapes in turn: the tables that hold a thread's plans
keep them all, so a query costs the same among 200 shapes as among 8."""
import ctypes
import time

import minitensor_amd as mt


def query(i):
    m, n, k = 64 + 13 * i, 96 + 29 * (i % 17), 512 + 7 * (i % 31)
    mats = [mt.MatF32(4096, 0, r, c, c, 1, 1, 0) for r, c in ((m, k), (k, n), (m, n))]
    return [ctypes.byref(x) for x in mats], mats   # (never read)


def seconds_per_query(shapes):
    f = mt.lib().mt_gemm_workspace_f32
    best = 1e9
    for _ in range(5):
        for args, _m in shapes:
            f(*args)
        t0 = time.perf_counter()
        for _ in range(2000 // len(shapes)):
            for args, _m in shapes:
                f(*args)
        best = min(best, (time.perf_counter() - t0) / (2000 // len(shapes) * len(shapes)))
    return best


def test_many_shapes_keep_their_plans():
    shapes = [query(i) for i in range(200)]
    few, many = seconds_per_query(shapes[:8]), seconds_per_query(shapes)
    # a shape that fell out of the tables is planned again, ten times a table's answer
    assert many < 3 * few, (few, many)
