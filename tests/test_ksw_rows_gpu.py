"""db out of the wave-split dW product of a Linear layer: row counts around a
chunk and a ring of them, widths off the tiles, both gradients accumulated."""
import numpy as np
import pytest
import torch

import minitensor_amd as mt
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [0, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("rows,fin,fout", [(1, 5, 3), (15, 33, 17), (64, 784, 130), (129, 63, 65),
                                           (1030, 40, 31)])
def test_db_from_the_wave_split_dw(dev, cfg, rows, fin, fout):
    x, dy = oracle.normal((rows, fin), 21), oracle.normal((rows, fout), 22)
    dw0, db0 = oracle.normal((fout, fin), 23), oracle.normal((fout,), 24)
    X, dY = torch.from_numpy(x).to(dev), torch.from_numpy(dy).to(dev)
    dw, db = torch.from_numpy(dw0).to(dev), torch.from_numpy(db0).to(dev)
    W = torch.zeros(fout, fin, device=dev)
    with mt.forced_config(mt.FAMILY_KSW, cfg, 1):
        mt.linear_backward(dY, X, W, need_dx=False, dw=dw, db=db, beta_w=1.0, beta_b=0.5)
        name = mt.last_config()
    # db out of this launch on 16x16 blocks (0: 32x32 ones, a launch of its own)
    assert name.startswith("ksw ") and f" cfg={cfg}" in name, name
    assert (" rows " in name) == (cfg != 0), name
    x64, y64 = x.astype(np.float64), dy.astype(np.float64)
    # rows + 2 roundings of 2^-24, each of at most the sum of the magnitudes
    eps = (rows + 2) * 2.0 ** -24
    want, mag = 0.5 * db0 + y64.sum(0), 0.5 * np.abs(db0) + np.abs(y64).sum(0)
    assert (np.abs(db.double().cpu().numpy() - want) <= eps * mag).all()
    want, mag = dw0 + y64.T @ x64, np.abs(dw0) + np.abs(y64).T @ np.abs(x64)
    assert (np.abs(dw.double().cpu().numpy() - want) <= eps * mag).all()
