"""db out of the weight gradient's launch is no further from 64 bits than the
launch of its own that it replaces."""
import pytest
import torch

import minitensor_amd as mt

pytestmark = pytest.mark.gpu


# (n, c, h, c_out, k, stride, pad): the stem, whose 401408 pixels are cut into 512
# ranges, and a layer of 64 ranges of 392
@pytest.mark.parametrize("layer", [(32, 3, 224, 64, 7, 2, 3), (32, 64, 28, 64, 3, 1, 1)])
def test_db_error(dev, layer):
    n, c, h, co, k, s, p = layer
    ho = (h + 2 * p - k) // s + 1
    g = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn(n, c, h, h, device=dev, generator=g)
    w = torch.zeros(co, c, k, k, device=dev)
    fused = alone = 0.0
    for _ in range(8):
        dy = torch.randn(n, co, ho, ho, device=dev, generator=g) * 0.01
        want = dy.double().sum((0, 2, 3))
        with mt.forced_config(mt.FAMILY_DL, 0, 64):
            db = mt.conv2d_backward(x, w, dy, s, p, need_dx=False)[2]
        assert " rows " in mt.last_config(), mt.last_config()   # db came out of the dW launch
        fused += float((db.double() - want).pow(2).sum())
        db = mt.conv2d_backward(x, w, dy, s, p, need_dx=False, need_dw=False)[2]
        alone += float((db.double() - want).pow(2).sum())
    assert fused <= alone, ((fused / alone) ** 0.5, mt.last_config())
