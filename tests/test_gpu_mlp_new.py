"""A network that was just created has parameters of zero, in every copy of
the weights that a kernel reads, also where the memory held another network's
before."""
import numpy as np
import pytest

from tests.test_mlp import small_net

pytestmark = pytest.mark.gpu


def used_and_closed(dims):
    """A network of the same sizes, its weights in every copy, given back."""
    from monte_carlompi_amd.mlp import Mlp
    n_in, H, L, n_out, batch = dims
    net = Mlp(*dims)
    net.set_params(np.full(net.n_params, 0.5, np.float32))
    x = np.ones((batch, n_in), np.float32)
    net.set_dataset(x, np.ones((batch, n_out), np.float32))
    net.train_steps(np.arange(batch, dtype=np.int32), batch, np.ones(n_out), lr=1e-3)
    net.close()


@pytest.mark.parametrize('dims', [(9, 256, 4, 651, 256), (5, 256, 1, 1, 64), (9, 256, 10, 100, 64), (9, 128, 3, 70, 64)])
def test_new_network_is_zero(monkeypatch, dims):
    import torch
    from monte_carlompi_amd._lib import MCS_FEATURES_IDENTITY
    from monte_carlompi_amd.mlp import Mlp
    n_in, H, L, n_out, batch = dims
    monkeypatch.setenv('MCS_MLP_LAYERED', '0')
    used_and_closed(dims)
    rng = np.random.default_rng(1)
    x = rng.normal(size=(batch, n_in)).astype(np.float32)
    t = rng.normal(size=(batch, n_out)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n_out).astype(np.float32)
    net = Mlp(*dims)
    np.testing.assert_array_equal(net.get_params(), 0.0)
    np.testing.assert_array_equal(net.forward(x), 0.0)
    one = np.ones(n_out)
    net.set_serving(MCS_FEATURES_IDENTITY, one, 0 * one, 0 * one)
    y = torch.full((batch, n_out), -1.0, device='cuda')
    xd = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    net.serve(xd, batch, y)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(y.cpu().numpy(), 1.0)                      # exp(0) - 0
    g, loss = net.grads(x, t, w)
    assert abs(loss - np.sum(w * t.astype(float) ** 2) / batch) < 1e-5 * loss
    layers = net.unflatten(g)
    for W, c in layers[:-1]:
        np.testing.assert_array_equal(W, 0.0)
        np.testing.assert_array_equal(c, 0.0)
    np.testing.assert_array_equal(layers[-1][0], 0.0)                       # silu(0) is 0
    ref = -2.0 * w * t.astype(float).sum(0) / batch
    # dY rounds to BF16, 2^-9 each at most
    assert np.all(np.abs(layers[-1][1] - ref) <= 2.0 ** -8 * 2.0 * w * np.abs(t).sum(0) / batch)
    net.set_dataset(x, t)
    net.train_steps(np.arange(batch, dtype=np.int32), batch, w, lr=1e-3)
    p = net.unflatten(net.get_params())
    assert np.all(np.isfinite(net.get_params()))
    for W, c in p[:-1]:
        np.testing.assert_array_equal(W, 0.0)
    np.testing.assert_allclose(np.abs(p[-1][1]), 1e-3, rtol=1e-3)           # the first step is the rate's size
    net.close()


def test_no_buffers_for_kernels_that_never_run(monkeypatch):
    """The row kernels' network at the largest batch: inputs 7 MB, targets
    and outputs 184 + 171, gradients of both 92, pre-activations and activations
    4 x (67 + 34), parameters and their sums 40: 0.90 GB.  The per-layer kernels'
    outputs and gradients (0.26 GB) are not among it."""
    import torch
    from monte_carlompi_amd.mlp import Mlp
    used = {}
    for layered in ('0', '1'):
        monkeypatch.setenv('MCS_MLP_LAYERED', layered)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        net = Mlp(9, 256, 4, 651, 65536)
        used[layered] = free - torch.cuda.mem_get_info()[0]
        net.close()
    print('bytes', used)
    assert 0.8e9 < used['0'] < 0.98e9
