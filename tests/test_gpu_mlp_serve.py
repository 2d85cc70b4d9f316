"""Inference of 256-wide networks (k_mlp_serve): bit for bit the per-layer
kernels' results around the row counts where the rows per block change and at
the edges of blocks, for shallow and deep networks and narrow and wide outputs,
features or raw case inputs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n_in,L,n_out,rows', [
    (9, 4, 651, (1, 31, 32, 33, 8192, 8193, 32768, 32769)), (1, 1, 1, (1, 257)), (32, 2, 64, (64, 8300)),
    (5, 16, 65, (100, 33000)), (3, 3, 1100, (63, 8200, 32900))])
def test_rows_and_shapes(monkeypatch, n_in, L, n_out, rows):
    import torch
    from monte_carlompi_amd import surrogate as S
    from monte_carlompi_amd._lib import MCS_FEATURES_IDENTITY, MCS_FEATURES_SNOW_BRF
    from monte_carlompi_amd.mlp import Mlp
    rng = np.random.default_rng(n_out)
    snow = n_in == S.N_FEAT
    nets = []
    for layered in ('0', '1'):
        monkeypatch.setenv('MCS_MLP_LAYERED', layered)
        net = Mlp(n_in, 256, L, n_out, max_batch=8192)
        net.init_params(seed=3)
        net.set_serving(MCS_FEATURES_SNOW_BRF if snow else MCS_FEATURES_IDENTITY, np.linspace(0.1, 1, n_out),
                        np.linspace(-1, 1, n_out), np.full(n_out, 1e-3), S.FEAT_MU if snow else None,
                        S.FEAT_SD if snow else None)
        nets.append(net)
    for n in rows:
        x = S.sample_inputs(n, n).astype(np.float32) if snow else rng.normal(size=(n, n_in)).astype(np.float32)
        q = torch.from_numpy(x).cuda()
        out = []
        for net in nets:
            y = torch.full((n + 1, n_out), -7.0, device='cuda')      # a row past the answers
            torch.cuda.synchronize()
            net.serve(q, n, y)
            assert bool((y[n] == -7.0).all())
            out.append(y[:n].cpu().numpy())
        np.testing.assert_array_equal(out[0], out[1])
        z = rng.normal(size=(min(n, 9000), n_in)).astype(np.float32)
        np.testing.assert_array_equal(nets[0].forward(z), nets[1].forward(z))
    for net in nets:
        net.close()
