"""A training step on the GPU against the layer-by-layer gradient and an Adam step in float64.

The two-launch step takes up to three hidden layers of 64 or 128; four layers (or wider ones) go
layer by layer, and both are held to the same bar.  The step's gradient has the rounding points of
`MLP.grad` (BF16 operands, FP32 sums), so what is left is FP32 rounding: in the sums and in Adam,
whose step is lr * m / (sqrt(v) + eps).  From the first step's gradient g the step is lr * sign(g)
for |g| >> 1e-8, so weights are compared where |g| > 1e-6 of its largest value:
|w - w_ref| <= 2^-23 |w| + 1e-4 lr.  The largest part of the 1e-4 is 1 - 0.999^t in FP32, 2^-24 / 0.002
= 3e-5 relative, half of that in its root."""
import numpy as np
import pytest

LR = 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("d_in,hidden,layers,d_out,batch", [
    (30, 128, 3, 3, 512),     # two ranges of rows in the weights' sums
    (1, 64, 1, 1, 64),        # the smallest
    (64, 64, 2, 16, 128),     # no padding in, every output column
    (65, 128, 1, 5, 320),     # one column past a padded width, one range
    (128, 64, 3, 2, 576),     # ranges of unequal length
    (128, 128, 2, 3, 16448),  # the most ranges, ragged
    (30, 64, 4, 3, 192),      # layer by layer
])
def test_training_step_is_adam_on_the_gradient(d_in, hidden, layers, d_out, batch):
    from nbodygo_amd.mlp import MLP
    rng = np.random.default_rng(batch + d_in)
    x = rng.normal(size=(batch, d_in)).astype(np.float32)
    t = rng.normal(size=(batch, d_out)).astype(np.float32)
    with MLP(d_in, hidden, layers, d_out, seed=7) as m:
        m1 = m2 = 0.0
        for step in range(1, 4):
            w = m.get_params().astype(np.float64)
            g32, loss = m.grad(x, t)
            g = g32.astype(np.float64)
            got_loss = m.train(x, t, steps=1, batch=batch, lr=LR)
            assert abs(got_loss - loss) <= 1e-5 * loss
            m1 = 0.9 * m1 + 0.1 * g
            m2 = 0.999 * m2 + 0.001 * g * g
            ref = w - LR * (m1 / (1 - 0.9 ** step)) / (np.sqrt(m2 / (1 - 0.999 ** step)) + 1e-8)
            got = m.get_params().astype(np.float64)
            big = np.abs(g) > 1e-6 * np.abs(g).max()
            assert big.any()
            err = np.abs(got - ref)[big]
            assert np.all(err <= 2.0 ** -23 * np.abs(ref[big]) + 1e-4 * LR), (step, err.max())
        # the weights that inference and the next forward read are the new ones
        np.testing.assert_array_equal(m.infer(x) if layers <= 3 else m.forward(x), m.forward(x))
