"""The two-launch training step has the bits of the layer-by-layer one: its products, sums and
roundings are the layer-by-layer gradient's (`MLP.grad` goes that way) and Adam's in FP32, in that
order, so weights and biases after several steps equal Adam in numpy's float32 on that gradient."""
import ctypes
import ctypes.util

import numpy as np
import pytest

f32 = np.float32
_m = ctypes.CDLL(ctypes.util.find_library("m"))
_m.powf.restype = ctypes.c_float
_m.powf.argtypes = [ctypes.c_float, ctypes.c_float]


def _adam(w, m1, m2, g, step, lr):
    """k_adam's expressions, operation by operation."""
    b1, b2, one = f32(0.9), f32(0.999), f32(1)
    c1 = one - f32(_m.powf(b1, step))
    c2 = one - f32(_m.powf(b2, step))
    m1 = b1 * m1 + (one - b1) * g
    m2 = b2 * m2 + (one - b2) * g * g
    return w - f32(lr) * (m1 / c1) / (np.sqrt(m2 / c2) + f32(1e-8)), m1, m2


@pytest.mark.gpu
@pytest.mark.parametrize("d_in,hidden,layers,d_out,batch", [
    (30, 128, 3, 3, 512),
    (1, 64, 1, 1, 64),
    (64, 64, 2, 16, 128),
    (65, 128, 1, 5, 320),
    (128, 64, 3, 2, 576),
    (128, 128, 2, 3, 16448),
    (30, 64, 4, 3, 192),      # layer by layer
])
def test_steps_are_adam_on_the_layer_by_layer_gradient(d_in, hidden, layers, d_out, batch):
    from nbodygo_amd.mlp import MLP
    rng = np.random.default_rng(batch + d_in)
    x = rng.normal(size=(batch, d_in)).astype(f32)
    t = rng.normal(size=(batch, d_out)).astype(f32)
    with MLP(d_in, hidden, layers, d_out, seed=7) as m:
        m1 = m2 = np.zeros(m.n_params, f32)
        w = m.get_params()
        for step in range(1, 6):
            g, _ = m.grad(x, t)
            w, m1, m2 = _adam(w, m1, m2, g, step, 1e-3)
            m.train(x, t, steps=1, batch=batch, lr=1e-3)
            assert w.dtype == f32
            np.testing.assert_array_equal(m.get_params(), w, err_msg="step %d" % step)
            # the fused inference reads transposed weights, kept by the two-launch step and made
            # again after the layer-by-layer one
            np.testing.assert_array_equal(m.infer(x), m.forward(x), err_msg="step %d" % step)
