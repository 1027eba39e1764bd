"""GPU: an image whose rows are longer than 32-bit byte offsets reach (2^25
columns and more, 64 channels of two and four bytes), forward and backward,
against the same columns cut out of it: around column 2^24, around 2^25, and
the first ones."""
import numpy as np
import pytest

import cnn_oracle as co
from hydist_amd import cnn

pytestmark = pytest.mark.gpu

L, CUT, NEAR = 3, 300, 100


def network(W, batch, ps):
    net = cnn.Network(1, W, batch=batch, layers=L)
    for l, (w, b) in enumerate(ps):
        net.set_layer(l, w, b)
    return net


def test_rows_past_32_bit_offsets():
    W = (1 << 25) + 170
    at = [0, (1 << 24) - CUT // 2, (1 << 25) - CUT // 2]
    rng = np.random.default_rng(8)
    ps = co.random_params(L, seed=9, scale=1.5)
    x = np.zeros((1, 1, W, 8), np.float32)
    tgt, msk = np.zeros((1, 1, W, 3), np.float32), np.zeros((1, 1, W), np.float32)
    cut = np.zeros((3, 1, CUT, 8), np.float32)
    cut_t, cut_m = np.zeros((3, 1, CUT, 3), np.float32), np.zeros((3, 1, CUT), np.float32)
    for k, a in enumerate(at):
        cut[k] = rng.normal(size=cut[k].shape)
        cut_t[k] = cut[k, ..., :3] + 0.2 * rng.normal(size=cut_t[k].shape)
        cut_m[k, 0, CUT // 2 - NEAR // 2:CUT // 2 + NEAR // 2] = 1
        x[0, :, a:a + CUT], tgt[0, :, a:a + CUT], msk[0, :, a:a + CUT] = cut[k], cut_t[k], cut_m[k]
    cut_m[0, 0, :NEAR] = msk[0, 0, :NEAR] = 1
    net = network(W, 1, ps)
    net.load(x, tgt, msk)
    pred = net.forward()
    loss = net.backward()
    grads = [net.get_grad(l) for l in range(L)]
    net.close()

    ref = network(CUT, 3, ps)
    ref.load(cut, cut_t, cut_m)
    want = ref.forward()
    for k, a in enumerate(at):
        inner = slice(0 if a == 0 else L, CUT - L)     # a cut's end columns see other neighbours
        assert np.array_equal(pred[0, 0, a:a + CUT][inner], want[k, 0][inner]), a
    assert np.abs(pred[0, 0, CUT:2 * CUT]).max() < np.abs(want).max()
    assert abs(loss / ref.backward() - 1.0) <= 1e-6
    for l in range(L):
        for got, w in zip(grads[l], ref.get_grad(l)):
            assert np.linalg.norm(got - w) <= 1e-5 * np.linalg.norm(w), l
    ref.close()
