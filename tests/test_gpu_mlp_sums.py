"""The gradient sums of 256-wide networks' training kernels have the addends of
the per-layer kernels: chunks of the batch, each one chain of MFMAs, and only
the order in which the chunks are added may differ.

With 64 rows every weight has two chunks, whose sum does not depend on the
order: the weight gradients, and the weights after an Adam step, are equal bit
for bit.  A lost or doubled term, an operand rounded at another place or other
chunks show there.  With more rows each of the up to 128 additions rounds by at
most 2^-24 of a running sum, ~sqrt(128) 2^-24 / 2 = 3e-7 relative for the array
in random order: 1e-6.  Biases are sums over rows in another order even at 64
(FP64 here, FP32 there): ~sqrt(64) 2^-24 = 5e-7 for addends of either sign:
1e-6."""
import numpy as np
import pytest

from tests.test_gpu_mlp_train import nets
from tests.test_mlp import small_net

pytestmark = pytest.mark.gpu


def off(u, v):
    return np.linalg.norm(u.astype(float) - v) / np.linalg.norm(v.astype(float))


def inputs(n_in, L, n_out, rows):
    rng = np.random.default_rng(rows + 10 * L + n_out)
    return (small_net(rng, n_in, 256, L, n_out), rng.normal(size=(rows, n_in)).astype(np.float32),
            (rng.normal(size=(rows, n_out)) * 0.5).astype(np.float32), rng.uniform(0.5, 1.5, n_out).astype(np.float32))


@pytest.mark.parametrize('n_in,L,n_out', [(9, 4, 651), (1, 1, 1), (32, 2, 64), (5, 3, 65), (9, 8, 1024), (7, 6, 200)])
def test_two_chunks_are_bitwise_the_per_layer_sums(monkeypatch, n_in, L, n_out):
    layers, x, t, w = inputs(n_in, L, n_out, 64)
    a, b = nets(monkeypatch, (n_in, 256, L, n_out, 64), layers)
    (ga, la), (gb, lb) = a.grads(x, t, w), b.grads(x, t, w)
    assert abs(la - lb) < 1e-6 * lb
    for l, ((Wa, ca), (Wb, cb)) in enumerate(zip(a.unflatten(ga), b.unflatten(gb))):
        np.testing.assert_array_equal(Wa, Wb, err_msg='layer %d' % l)
        assert off(ca, cb) < 1e-6, l
    for net in (a, b):
        net.set_dataset(x, t)
        net.train_steps(np.arange(64, dtype=np.int32), 64, w, lr=1e-3, weight_decay=1e-3)
    for l, ((Wa, ca), (Wb, cb)) in enumerate(zip(a.unflatten(a.get_params()), b.unflatten(b.get_params()))):
        np.testing.assert_array_equal(Wa, Wb, err_msg='layer %d' % l)
    a.close(); b.close()


@pytest.mark.parametrize('n_in,L,n_out,batch', [(9, 4, 651, 4096), (32, 2, 64, 128), (5, 3, 65, 192), (9, 8, 1024, 1088),
                                                (9, 5, 129, 320), (3, 6, 200, 576), (7, 7, 33, 640), (9, 1, 1000, 8192)])
def test_chunks_in_another_order_only(monkeypatch, n_in, L, n_out, batch):
    layers, x, t, w = inputs(n_in, L, n_out, batch)
    a, b = nets(monkeypatch, (n_in, 256, L, n_out, batch), layers)
    (ga, la), (gb, lb) = a.grads(x, t, w), b.grads(x, t, w)
    assert abs(la - lb) < 1e-6 * lb
    for l, ((Wa, ca), (Wb, cb)) in enumerate(zip(a.unflatten(ga), b.unflatten(gb))):
        assert off(Wa, Wb) < 1e-6 and off(ca, cb) < 1e-6, (l, off(Wa, Wb), off(ca, cb))
    a.close(); b.close()


@pytest.mark.parametrize('n_in,L,n_out', [(9, 4, 651), (5, 1, 65)])
def test_adam_with_moments_rounds_as_the_per_layer_path(monkeypatch, n_in, L, n_out):
    """The first steps with a learning rate of zero fill the moments from
    gradients that both paths have bit for bit (the parameters stay); the step
    after them then gives the same weights only if the moments' expressions
    round alike."""
    layers, x, t, w = inputs(n_in, L, n_out, 256)
    nets_ = nets(monkeypatch, (n_in, 256, L, n_out, 64), layers)
    got = []
    for net in nets_:
        net.set_dataset(x, t)
        idx = np.arange(256, dtype=np.int32)
        net.train_steps(idx[:192], 64, w, lr=0.0)
        np.testing.assert_array_equal(net.get_params(), net.flatten(layers))
        net.train_steps(idx[192:], 64, w, lr=1e-2, weight_decay=1e-2)
        got.append(net.unflatten(net.get_params()))
    for l, ((Wa, ca), (Wb, cb), (W0, c0)) in enumerate(zip(*got, layers)):
        np.testing.assert_array_equal(Wa, Wb, err_msg='layer %d' % l)
        assert np.mean(Wa != W0) > 0.9
    for net in nets_:
        net.close()
