"""GPU: hd_cnn_backward differentiates the last forward pass, also where that
was a prediction into a context (hd_cnn_predict_into_ctx): the gradients are
those of a network that was given the context's image from the host."""
import numpy as np
import pytest

import cnn_oracle as co
from hydist_amd import cnn, synth
from hydist_amd._lib import Solver

pytestmark = pytest.mark.gpu

SCALES = dict(s_u=1.0, s_v=1.0, s_z=1.0, s_b=1e30, s_q=500.0, s_h=10.0, d_u=0.5, d_v=0.5, d_z=0.5)
L = 4


def network(H, W, ps):
    net = cnn.Network(H, W, batch=1, layers=L)
    net.set_scales(**SCALES)
    net.set_sparse(False)
    for l, (w, b) in enumerate(ps):
        net.set_layer(l, w, b)
    return net


def test_backward_after_a_prediction():
    c = synth.channel_case(N=20, M=37, nsteps=10)
    g = Solver(c)
    g.init()
    rng = np.random.default_rng(4)
    shape = (c.N + 3, c.M + 3)
    for n in ("u", "v", "z"):
        g.set(n, 0.5 * rng.standard_normal(shape))
    q, zb = 300.0, 0.25
    wet = g.get("khouot") == 0
    x8 = np.zeros((1,) + shape + (8,), np.float32)
    for k, n in enumerate(("u", "v", "z")):
        x8[0, ..., k] = np.where(wet, g.get(n), 0.0)
    x8[0, ..., 4] = wet
    x8[0, ..., 5], x8[0, ..., 6] = np.float32(q) / np.float32(500.0), zb
    x8[0, ..., 7] = g.get("h") / 10.0
    tgt = (x8[..., :3] + 0.3 * rng.standard_normal((1,) + shape + (3,))).astype(np.float32)
    msk = wet[None].astype(np.float32)

    ps = co.random_params(L, seed=5, scale=1.5)
    a, b = network(*shape, ps), network(*shape, ps)
    other = rng.normal(size=x8.shape).astype(np.float32)
    a.load(other, tgt, msk)
    a.forward()
    a.predict_into(g, q, zb)
    b.load(x8, tgt, msk)
    b.forward()
    # the same pass; the weight gradients' sums differ in their order
    assert abs(a.backward() / b.backward() - 1.0) <= 1e-6
    for l in range(L):
        for got, want in zip(a.get_grad(l), b.get_grad(l)):
            assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want), l
    a.close()
    b.close()
