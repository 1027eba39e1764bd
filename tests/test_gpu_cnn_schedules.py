"""GPU: the network's convolutions and weight gradients where a workgroup takes
more than one item and items have more rows than the smallest schedule's four:
1024 items of 33 rows on 512 workgroups (tall narrow images, the last item of
a column shorter), three items to some, odd and even rows an item.  Against
the CPU restatement on the same bfloat16 activations and weights.  Tolerances:
1 % of the output's scale forward; backward 2 % of a layer's gradient norm
(the gradient images are rounded to bfloat16, 2^-9, once a layer, three times
here; the rest is for activations that round the other way)."""
import numpy as np
import pytest

import cnn_oracle as co
from hydist_amd import cnn
from test_gpu_cnn_shapes import grads_at

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,nimg", [(2100, 5, 16), (2087, 3, 17), (1850, 2, 40), (8200, 1, 13), (251, 268, 1),
                                      (1390, 33, 12)])
def test_forward_and_gradients(H, W, nimg):
    L = 3
    rng = np.random.default_rng(H + W)
    ps = [(w.astype(np.float32).astype(np.float64), b.astype(np.float32).astype(np.float64))
          for w, b in co.random_params(L, seed=H, scale=1.5)]
    net = cnn.Network(H, W, batch=nimg, layers=L)
    for l, (w, b) in enumerate(ps):
        net.set_layer(l, w, b)
    x8 = rng.normal(size=(nimg, H, W, 8)).astype(np.float32)
    tgt = (x8[..., :3] + 0.2 * rng.normal(size=(nimg, H, W, 3))).astype(np.float32)
    msk = (rng.random((nimg, H, W)) > 0.25).astype(np.float32)
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
