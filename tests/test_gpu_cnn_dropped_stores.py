"""GPU: the last layer's lanes that hold padded output channels store nothing:
with weights and biases in those channels, too, the prediction has the bits
that it has without, at the first columns of a row above all."""
import numpy as np
import pytest

import cnn_oracle as co
from hydist_amd import cnn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W", [(1, 1), (6, 2), (5, 16), (4, 64), (9, 65), (3, 130)])
def test_padded_channels_leave_no_trace(H, W):
    L = 3
    rng = np.random.default_rng(W)
    ps = co.random_params(L, seed=W, scale=1.5)
    x = rng.normal(size=(2, H, W, 8)).astype(np.float32)
    preds = []
    for padded in (False, True):
        net = cnn.Network(H, W, batch=2, layers=L)
        for l, (w, b) in enumerate(ps):
            w, b = w.copy(), b.copy()
            if padded and l == L - 1:
                w[:, co.COUT:] = 50.0 + rng.random(w[:, co.COUT:].shape)
                b[co.COUT:] = -1000.0
            net.set_layer(l, w, b)
        net.load(x)
        preds.append(net.forward())
        net.close()
    assert np.array_equal(preds[0], preds[1])
