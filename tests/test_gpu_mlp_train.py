"""The fused training step (weight gradients straight into Adam, BF16 weight
copies and their transposes rewritten by the same kernel) against Adam in numpy
on the gradients of ``Ensemble.gradients``, at widths and batches around the
64-entry tiles.

Both sides use the same FP32 gradients (same kernel, same order of sums), so a
step differs by the rounding of Adam's own FP32 arithmetic: a few ulp (6e-8) of
the update, whose size is at most lr, and one ulp of the weight.  The second
step's gradients come from a network loaded with the first step's weights: a
stale BF16 copy or transpose would change them in the third digit.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,batch", [((8, 64, 64, 64), 64), ((8, 72, 40, 100), 37), ((5, 65, 63, 129, 1), 1),
                                        ((8, 128, 130), 65), ((3, 7), 130), ((64, 200, 64), 200)])
def test_fused_adam_steps_match_numpy(gpu, dims, batch):
    from impuritymodel_amd.surrogate import Ensemble

    E, lr, b1, b2, eps = 2, np.float32(1e-2), np.float32(0.9), np.float32(0.999), np.float32(1e-8)
    rng = np.random.default_rng(11)
    x = rng.uniform(-1, 1, (batch, dims[0])).astype(np.float32)
    t = rng.normal(size=(batch, dims[-1])).astype(np.float32)
    net, probe = Ensemble(E, dims, max_batch=8, seed=3), Ensemble(E, dims, max_batch=8, seed=3)
    p0 = net.init_params(9) + rng.normal(0, 0.01, (E, net.P)).astype(np.float32)
    used = sum(dims[l + 1] * (dims[l] + 1) for l in range(len(dims) - 1))
    p0[:, used:] = 0.0
    net.set_params(p0)
    losses = net.train(x, t, epochs=2, batch=batch, lr=float(lr), seed=4)
    p = p0.copy()
    m, v = np.zeros_like(p), np.zeros_like(p)
    for step in (1, 2):
        probe.set_params(p)
        # the second step's rows are another permutation of the same batch; the
        # gradients then differ by the order of an FP32 sum over the batch
        rows = np.random.default_rng(4)
        for _ in range(step):
            order = rows.permutation(batch)
        loss, g = probe.gradients(x[order], t[order])
        np.testing.assert_allclose(losses[step - 1], loss, rtol=1e-5)
        m = b1 * m + (np.float32(1) - b1) * g
        v = b2 * v + (np.float32(1) - b2) * g * g
        bc1, bc2 = np.float32(1) - b1 ** step, np.float32(1) - b2 ** step
        p = p - lr * (m / bc1) / (np.sqrt(v / bc2) + eps)
    got = net.get_params()
    assert np.array_equal(got[:, used:], p0[:, used:])
    # an update is lr m'/(sqrt(v') + eps): where |g| is near eps its relative
    # error is that of the gradient, elsewhere a few ulp; 1e-5 of lr holds both
    assert np.quantile(np.abs(got - p), 0.999) <= 1e-5 * lr + 2e-7 * np.abs(p).max()
    assert np.abs(got - p).max() <= 2e-2 * lr
