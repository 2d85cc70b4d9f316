"""Serving more rows than one launch can hold."""
import numpy as np
import pytest

from tests.test_mlp import small_net

pytestmark = pytest.mark.gpu


def test_more_rows_than_a_launch_has_threads(monkeypatch):
    """1025 times the same 2^20 queries (4.3 GB in, 4.3 GB out): past 2^30 rows
    a single launch would need over 2^32 threads.  Every copy is answered as
    the first alone."""
    import torch
    from monte_carlompi_amd._lib import MCS_FEATURES_IDENTITY
    from monte_carlompi_amd.mlp import Mlp
    monkeypatch.setenv('MCS_MLP_LAYERED', '0')
    rng = np.random.default_rng(3)
    net = Mlp(1, 256, 1, 1, max_batch=64)
    net.set_params(Mlp.flatten(small_net(rng, 1, 256, 1, 1)))
    net.set_serving(MCS_FEATURES_IDENTITY, np.ones(1), np.zeros(1), np.zeros(1))
    q, k = 1 << 20, 1025
    x = torch.randn(q, 1, device='cuda', generator=torch.Generator('cuda').manual_seed(1))
    one = torch.empty(q, 1, device='cuda')
    xs = x.repeat(k, 1)
    y = torch.full((k * q, 1), -1.0, device='cuda')
    torch.cuda.synchronize()
    net.serve(x, q, one)
    net.serve(xs, k * q, y)
    torch.cuda.synchronize()
    assert one.std() > 0
    for a in range(0, k, 41):
        assert torch.equal(y.view(k, q)[a:a + 41], one.view(1, q).expand(41, q)), a
    net.close()
