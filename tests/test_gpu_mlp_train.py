"""Training of 256-wide networks (k_train_rows, k_train_dw, k_train_adam)
against the per-layer kernels and the float64 reference.

Tolerances.  Both paths round the same quantities to bf16 and accumulate in
FP32; they add in different orders, so sums differ by ~sqrt(K) 2^-24 relative
and a bf16 rounding flips where the sum lies that close to a tie: a share of
about 2^-24 sqrt(256) / 2^-9 = 5e-4 of the elements, each by 2^-8, an rms of
1e-4 relative per layer.  Gradients of the two paths are compared at 2e-3
(10 x over two layers' worth).  Against float64 on bf16-rounded weights the
path's own bf16 rounding of activations and gradients (2^-9 rms each, up to
nine of them) gives ~1e-2; the bound is the one the per-layer kernels have,
3e-2."""
import numpy as np
import pytest

from tests import mlp_ref
from tests.test_mlp import bf16_round, small_net

pytestmark = pytest.mark.gpu


def nets(monkeypatch, dims, layers):
    from monte_carlompi_amd.mlp import Mlp
    out = []
    for layered in ('0', '1'):
        monkeypatch.setenv('MCS_MLP_LAYERED', layered)
        net = Mlp(*dims)
        net.set_params(Mlp.flatten(layers))
        out.append(net)
    return out


@pytest.mark.parametrize('n_in,L,n_out,batch', [(9, 4, 651, 4096), (1, 1, 1, 64), (32, 2, 64, 128), (5, 3, 65, 192),
                                                (9, 8, 1024, 1088), (9, 5, 129, 64), (3, 6, 200, 576), (7, 7, 33, 640)])
def test_gradients(monkeypatch, n_in, L, n_out, batch):
    rng = np.random.default_rng(batch + L)
    layers = small_net(rng, n_in, 256, L, n_out)
    a, b = nets(monkeypatch, (n_in, 256, L, n_out, batch), layers)
    x = rng.normal(size=(batch, n_in)); t = rng.normal(size=(batch, n_out)) * 0.5
    w = rng.uniform(0.5, 1.5, n_out)
    (ga, la), (gb, lb) = a.grads(x, t, w), b.grads(x, t, w)
    assert abs(la - lb) < 1e-3 * lb
    lref = [(bf16_round(W), c) for W, c in layers]
    loss, gref = mlp_ref.loss_and_grads(lref, bf16_round(x), t, w)
    assert abs(la - loss) < 2e-2 * loss
    for (Wa, ca), (Wb, cb), (Wr, cr) in zip(a.unflatten(ga), b.unflatten(gb), gref):
        for u, v, r in ((Wa, Wb, Wr), (ca, cb, cr)):
            assert np.linalg.norm(u - v) < 2e-3 * np.linalg.norm(v)
            assert np.linalg.norm(u - r) < 3e-2 * np.linalg.norm(r)
    g2, l2 = a.grads(x, t, w)
    np.testing.assert_array_equal(ga, g2)             # no atomics: the same sums every time
    assert la == l2
    a.close(); b.close()


def test_training_and_inference_after_it(monkeypatch):
    """Adam steps follow the per-layer path's; inference then uses the trained
    weights; a network set anew starts from clean moments; smaller batches
    after larger ones."""
    rng = np.random.default_rng(3)
    n_in, n_out, n = 9, 130, 3000
    layers = small_net(rng, n_in, 256, 3, n_out)
    a, b = nets(monkeypatch, (n_in, 256, 3, n_out, 1024), layers)
    x = rng.normal(size=(n, n_in))
    t = np.tanh(x @ rng.normal(size=(n_in, n_out))) * 0.5
    w = np.full(n_out, 1.0 / n_out)
    idx = rng.integers(0, n, 5 * 1024)
    losses = []
    for net in (a, b):
        net.set_dataset(x, t)
        ls = [net.train_steps(idx, 1024, w, lr=1e-3, weight_decay=1e-3), net.train_steps(idx[:3 * 64], 64, w, lr=1e-3)]
        losses.append(np.concatenate(ls))
    np.testing.assert_allclose(losses[0], losses[1], rtol=5e-3)
    assert losses[0][4] < losses[0][0]
    pa, pb, p0 = a.get_params(), b.get_params(), a.flatten(layers)
    # eight Adam steps of ~1e-3 each: the updates agree to the noise of the gradients' signs near zero
    assert np.linalg.norm(pa - pb) < 0.1 * np.linalg.norm(pb - p0)
    ya, yb = a.forward(x), b.forward(x)
    assert np.linalg.norm(ya - yb) < 2e-2 * np.linalg.norm(yb)
    c = type(a)(n_in, 256, 3, n_out, 1024)
    c.set_params(pa)
    monkeypatch.setenv('MCS_MLP_LAYERED', '0')
    np.testing.assert_array_equal(c.forward(x), ya)     # the bf16 copies are those of the FP32 parameters
    a.set_params(a.flatten(layers))
    np.testing.assert_array_equal(a.train_steps(idx, 1024, w, lr=1e-3, weight_decay=1e-3), losses[0][:5])
    for net in (a, b, c):
        net.close()
