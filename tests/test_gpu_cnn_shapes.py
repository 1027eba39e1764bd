"""GPU: the network's convolutions and weight gradients at image sizes around
their strips (16, 32 and 64 columns) and row blocks, against the CPU
restatement on the same bfloat16 activations and weights.  Tolerances: 1 % of
the output's scale forward; backward 2 % of a layer's gradient norm (the
gradient images are rounded to bfloat16, 2^-9, once a layer, four times
here; the rest is for activations that round the other way)."""
import numpy as np
import pytest

import cnn_oracle as co
from hydist_amd import cnn

pytestmark = pytest.mark.gpu


def grads_at(params, x8, tgt, msk):
    """Loss and gradients of the masked MSE in FP64, the weights, activations
    and ReLU gates being the BF16 ones of the emulated forward pass."""
    pred, c = co.forward(params, x8, emulate_bf16=True)
    acts, rels, Ws = c["acts"], c["rels"], c["Ws"]
    L = len(params)
    norm = 3.0 * msk.sum()
    d = pred - tgt
    dout = np.zeros(c["out"].shape)
    dout[..., :co.COUT] = 2.0 * msk[..., None] * d / norm
    grads = [None] * L
    dA, dZ = None, dout
    for l in range(L - 1, -1, -1):
        grads[l] = (co.conv_wgrad(acts[l], dZ), dZ.sum(axis=(0, 1, 2)))
        if l == 0:
            break
        back = co.conv_dgrad(dZ, Ws[l])
        dA = back if dA is None else dA + back
        dZ = dA * ((rels[l - 1] if l > 1 else acts[1]) > 0)
    return float((msk[..., None] * d * d).sum() / norm), grads


@pytest.mark.parametrize("H,W,nimg", [(1, 1, 1), (2, 15, 2), (3, 16, 2), (4, 17, 1), (5, 32, 1), (6, 33, 2), (70, 65, 1),
                                      (2, 131, 3)])
def test_forward_and_gradients(H, W, nimg):
    L = 4
    rng = np.random.default_rng(H * 1000 + W)
    ps = [(w.astype(np.float32).astype(np.float64), b.astype(np.float32).astype(np.float64))
          for w, b in co.random_params(L, seed=W, scale=1.5)]
    net = cnn.Network(H, W, batch=nimg, layers=L)
    for l, (w, b) in enumerate(ps):
        net.set_layer(l, w, b)
    x8 = rng.normal(size=(nimg, H, W, 8)).astype(np.float32)
    tgt = (x8[..., :3] + 0.2 * rng.normal(size=(nimg, H, W, 3))).astype(np.float32)
    msk = (rng.random((nimg, H, W)) > 0.25).astype(np.float32)
    msk[0, 0, 0] = 1
    net.load(x8, tgt, msk)
    pred = net.forward()
    ref, _ = co.forward(ps, x8.astype(np.float64), emulate_bf16=True)
    scale = np.abs(ref - x8[..., :3]).max()
    assert np.abs(pred - ref).max() <= 1e-2 * scale + 1e-4
    loss = net.backward()
    loss_ref, g = grads_at(ps, x8.astype(np.float64), tgt.astype(np.float64), msk.astype(np.float64))
    assert abs(loss - loss_ref) <= 2e-2 * loss_ref
    for l in range(L):
        dw, db = net.get_grad(l)
        for got, want in ((dw, g[l][0]), (db, g[l][1])):
            assert np.linalg.norm(got - want) <= 2e-2 * np.linalg.norm(want) + 1e-6, l
    net.close()
