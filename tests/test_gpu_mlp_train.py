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


def _layer_views(p, dims):
    """Views (weights [members, out, in], biases [members, out]) of flat parameters, by layer."""
    out, off = [], 0
    for l in range(len(dims) - 1):
        i, o = dims[l], dims[l + 1]
        out.append((p[:, off:off + o * i].reshape(len(p), o, i), p[:, off + o * i:off + o * i + o]))
        off += o * i + o
    return out


@pytest.mark.parametrize("dims", [(8, 100, 72, 70), (5, 100, 72, 70), (8, 64, 128, 64)])
def test_infinite_activations_stay_in_their_sample(gpu, dims):
    """One hidden unit of one sample overflows: with positive weights behind it every output of
    that sample is +inf (no product is inf * 0 or inf - inf), the other samples are those of the
    network without that unit's weight, bit for bit."""
    from impuritymodel_amd.surrogate import Ensemble

    net = Ensemble(2, dims, max_batch=8, seed=3)
    plain = np.abs(net.init_params(9)) + np.float32(1e-3)
    plain[:, sum(dims[l + 1] * (dims[l] + 1) for l in range(3)):] = 0.0
    for _, b in _layer_views(plain, dims):
        b[:] = 0.0
    _layer_views(plain, dims)[0][0][:, 7, 0] = 0.0
    huge = plain.copy()
    _layer_views(huge, dims)[0][0][:, 7, 0] = 2.0 ** 127
    x = np.random.default_rng(2).uniform(0.1, 1, (6, dims[0])).astype(np.float32)
    x[:, 0] = 0.0
    net.set_params(plain)
    want = net.forward(x)
    x[2, 0] = 4.0
    net.set_params(huge)
    got = net.forward(x)
    keep = np.arange(6) != 2
    assert np.array_equal(got[:, keep], want[:, keep]) and np.all(np.isfinite(got[:, keep]))
    assert np.all(got[:, 2] == np.inf)
    # the same through the training pass: the sample's losses and gradients are not finite,
    # so it is the forward's other samples alone that can be compared: leave it out
    g0 = net.gradients(x[keep], want[0, keep])
    net.set_params(plain)
    g1 = net.gradients(x[keep], want[0, keep])
    assert np.array_equal(g0[0], g1[0]) and np.all(np.isfinite(g0[1]))
    for l, ((w0, b0), (w1, b1)) in enumerate(zip(_layer_views(g0[1], dims), _layer_views(g1[1], dims))):
        assert np.array_equal(w0, w1) and np.array_equal(b0, b1), l


@pytest.mark.parametrize("dims,batch", [((8, 100, 72, 70), 3), ((8, 64, 64, 64), 65)])
def test_gradients_with_overflow_in_the_padding_samples(gpu, dims, batch):
    """A bias of 2^127 that every sample cancels exactly: z = 0 for the batch, while the rows that
    pad the batch to whole tiles overflow in the second layer.  Losses and gradients are those of
    the network without the bias and the weight, bit for bit."""
    from impuritymodel_amd.surrogate import Ensemble

    net = Ensemble(2, dims, max_batch=8, seed=3)
    rng = np.random.default_rng(5)
    plain = net.init_params(9)
    views = _layer_views(plain, dims)
    views[0][0][:, 7, :] = 0.0
    views[0][1][:, 7] = 0.0
    views[1][0][:, :, 7] = 4.0
    big = plain.copy()
    views = _layer_views(big, dims)
    views[0][0][:, 7, 0] = -(2.0 ** 127)
    views[0][1][:, 7] = 2.0 ** 127
    x = rng.uniform(-1, 1, (batch, dims[0])).astype(np.float32)
    x[:, 0] = 1.0
    t = rng.normal(size=(batch, dims[-1])).astype(np.float32)
    net.set_params(plain)
    want_loss, want = net.gradients(x, t)
    net.set_params(big)
    loss, got = net.gradients(x, t)
    assert np.all(np.isfinite(want)) and np.array_equal(loss, want_loss) and np.array_equal(got, want)
    p = [net.train(x, t, epochs=1, batch=batch, lr=1e-3), net.get_params()]
    assert np.all(np.isfinite(p[0])) and np.all(np.isfinite(p[1]))


def test_losses_of_many_steps_in_one_call(gpu):
    """More steps in one call than the partial sums are kept for (256 at this size): the same
    losses and weights as in calls of 100 steps, bit for bit (constant learning rate)."""
    from impuritymodel_amd.surrogate import Ensemble

    rng = np.random.default_rng(8)
    x = rng.uniform(-1, 1, (512, 4)).astype(np.float32)
    t = rng.normal(size=(512, 2048)).astype(np.float32)
    out = []
    for chunk in (100, 600):
        net = Ensemble(2, (4, 2048), max_batch=512, seed=3)
        out.append((net.train(x, t, epochs=600, batch=512, lr=1e-3, seed=4, chunk=chunk), net.get_params()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert np.all(out[0][0] > 0) and np.all(out[0][0][-1] < out[0][0][0])
