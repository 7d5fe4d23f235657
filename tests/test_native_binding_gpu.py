"""The native binding of the Python calls against the same calls through ctypes:
bit for bit, on views, batches, accumulation and given outputs, and the same
errors."""
import pytest
import torch

import minitensor_amd as mt

pytestmark = pytest.mark.gpu


class Declined:
    """A binding that leaves every call to the Python path."""

    def __getattr__(self, name):
        return lambda *a, **k: None


class Recorded:
    """The binding, with what it answered."""

    def __init__(self, real, answers):
        self.real, self.answers = real, answers

    def __getattr__(self, name):
        def call(*a, **k):
            r = getattr(self.real, name)(*a, **k)
            self.answers.append(r)
            return r
        return call


def both(monkeypatch, call):
    answers, real = [], mt.native()
    with monkeypatch.context() as m:
        m.setattr(mt, "native", lambda: Recorded(real, answers))
        got = call()
    assert answers and all(r is not None for r in answers)   # it took the call
    with monkeypatch.context() as m:
        m.setattr(mt, "native", Declined)
        want = call()
    got, want = [r if isinstance(r, tuple) else (r,) for r in (got, want)]
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)


def rnd(dev, *shape, seed=1):
    g = torch.Generator(device="cpu").manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=g).to(dev)


CALLS = {
    "gemm": lambda d: mt.gemm(rnd(d, 65, 130), rnd(d, 130, 77)),
    "gemm_view": lambda d: mt.gemm(rnd(d, 70, 64)[3:], rnd(d, 40, 64).t(), bias=rnd(d, 40),
                                   bias_axis=mt.BIAS_COL),
    "gemm_steps": lambda d: mt.gemm(rnd(d, 64, 64)[::2, ::3], rnd(d, 22, 18)),
    "gemm_beta": lambda d: mt.gemm(rnd(d, 512, 300), rnd(d, 300, 256), out=rnd(d, 512, 256),
                                   bias=rnd(d, 512), bias_axis=mt.BIAS_ROW, beta=0.5),
    "bmm_broadcast": lambda d: mt.gemm(rnd(d, 1, 33, 20), rnd(d, 4, 20, 31)),
    "gemm_k0": lambda d: mt.gemm(rnd(d, 5, 0), rnd(d, 0, 6)),
    "gemm_empty": lambda d: mt.gemm(rnd(d, 0, 5), rnd(d, 5, 6)),
    "linear": lambda d: mt.linear(rnd(d, 33, 100), rnd(d, 70, 100), rnd(d, 70)),
    "linear_backward": lambda d: mt.linear_backward(rnd(d, 33, 70), rnd(d, 33, 100),
                                                    rnd(d, 70, 100)),
    "linear_accumulate": lambda d: mt.linear_backward(
        rnd(d, 64, 130), rnd(d, 64, 784), rnd(d, 130, 784), need_dx=False, dw=rnd(d, 130, 784),
        db=rnd(d, 130), beta_w=1.0, beta_b=1.0),
    "conv2d": lambda d: mt.conv2d(rnd(d, 2, 16, 9, 9), rnd(d, 24, 16, 3, 3), rnd(d, 24), padding=1),
    "conv2d_view": lambda d: mt.conv2d(rnd(d, 2, 9, 9, 16).permute(0, 3, 1, 2),
                                       rnd(d, 24, 16, 1, 1), stride=2),
    "conv2d_backward": lambda d: mt.conv2d_backward(rnd(d, 2, 6, 9, 9), rnd(d, 8, 6, 3, 3),
                                                    rnd(d, 2, 8, 5, 5), stride=2, padding=1),
}
BAD = {
    "inner": lambda d: mt.gemm(rnd(d, 3, 4), rnd(d, 5, 6)),
    "double": lambda d: mt.gemm(rnd(d, 3, 4).double(), rnd(d, 4, 6).double()),
    "cpu": lambda d: mt.gemm(rnd("cpu", 3, 4), rnd(d, 4, 6)),
    "out": lambda d: mt.gemm(rnd(d, 3, 4), rnd(d, 4, 6), out=rnd(d, 6, 3)),
    "bias": lambda d: mt.gemm(rnd(d, 3, 4), rnd(d, 4, 6), bias=rnd(d, 6)),
    "linear": lambda d: mt.linear(rnd(d, 3, 4), rnd(d, 5, 6)),
    "conv": lambda d: mt.conv2d(rnd(d, 1, 4, 5, 5), rnd(d, 3, 5, 3, 3)),
    "dy": lambda d: mt.conv2d_backward(rnd(d, 1, 4, 5, 5), rnd(d, 3, 4, 3, 3), rnd(d, 1, 3, 4, 4)),
}


@pytest.mark.parametrize("name", CALLS)
def test_same_results(dev, monkeypatch, name):
    both(monkeypatch, lambda: CALLS[name](dev))


@pytest.mark.parametrize("name", BAD)
def test_same_errors(dev, monkeypatch, name):
    with pytest.raises(Exception) as got:
        BAD[name](dev)
    monkeypatch.setattr(mt, "native", Declined)
    with pytest.raises(Exception) as want:
        BAD[name](dev)
    assert got.type is want.type and str(got.value) == str(want.value)
