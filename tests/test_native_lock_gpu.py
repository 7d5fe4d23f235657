"""The native calls let other Python threads run while they plan and launch."""
import sys
import threading
import time

import pytest
import torch

import minitensor_amd as mt

pytestmark = pytest.mark.gpu

CALLS = {
    "gemm": lambda t, n: (mt.gemm, t[:40, :n], t[:n, :50]),
    "linear": lambda t, n: (mt.linear, t[:40, :n], t[:50, :n]),
    "linear_backward": lambda t, n: (mt.linear_backward, t[:40, :50], t[:40, :n], t[:50, :n]),
    "conv2d": lambda t, n: (mt.conv2d, t.view(-1)[:n * 64].view(1, n, 8, 8),
                            t.view(-1)[:4 * n].view(4, n, 1, 1)),
    "conv2d_backward": lambda t, n: (mt.conv2d_backward, t.view(-1)[:n * 64].view(1, n, 8, 8),
                                     t.view(-1)[:4 * n].view(4, n, 1, 1),
                                     t.view(-1)[:256].view(1, 4, 8, 8)),
}


@pytest.mark.parametrize("name", CALLS)
def test_other_threads_run(dev, name):
    t = torch.zeros(1024, 1024, device=dev)
    # sizes that are new to the planner, so that a call takes longer; the arguments
    # beforehand, since making them gives the lock up too
    calls = [CALLS[name](t, n) for n in range(64, 964)]
    fn, *args = calls[0]
    fn(*args)
    steps, stop = [0], threading.Event()

    def count():
        while not stop.is_set():
            steps[0] += 1
            time.sleep(0)   # gives the lock back at once

    old = sys.getswitchinterval()
    sys.setswitchinterval(100)   # nobody is made to give it up
    thread = threading.Thread(target=count)
    try:
        thread.start()
        before, seen = steps[0], 0
        for fn, *args in calls:
            fn(*args)
            seen = steps[0] - before
            if seen:
                break
    finally:
        sys.setswitchinterval(old)
        stop.set()
        thread.join()
    assert seen, "no other thread ran during 900 calls"
