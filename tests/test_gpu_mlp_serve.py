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


def bf16_bits(x64, via_f32):
    """x64 rounded to BF16 (nearest even) in one step, or by way of float32;
    as float32 values."""
    f = x64.astype(np.float32)
    u = f.view(np.uint32).astype(np.int64)
    if not via_f32:
        # round to odd in float32 first: the second rounding then sees every
        # inexact bit
        lost = f.astype(np.float64) != x64
        away = lost & (np.abs(f.astype(np.float64)) > np.abs(x64))
        u = np.where(lost, (u - away) | 1, u)
    r = (u + 0x7FFF + ((u >> 16) & 1)) & ~np.int64(0xFFFF)
    return r.astype(np.uint32).view(np.float32)


@pytest.mark.parametrize('layered', ['0', '1'])
def test_first_feature_rounds_once(monkeypatch, layered):
    """r_eff whose standardised logarithm is a BF16 tie in float32 but not in
    float64: the first feature is rounded straight from float64.  A network that
    passes the feature through one SiLU unit shows which value it was."""
    import torch
    from monte_carlompi_amd import surrogate as S
    from monte_carlompi_amd._lib import MCS_FEATURES_SNOW_BRF
    from monte_carlompi_amd.mlp import Mlp
    monkeypatch.setenv('MCS_MLP_LAYERED', layered)
    rng = np.random.default_rng(0)
    reff = np.exp(rng.uniform(np.log(30.0), np.log(1500.0), 4_000_000)).astype(np.float32)
    mu, sd = np.float32(S.FEAT_MU[0]), np.float32(S.FEAT_SD[0])
    f = (np.log(reff.astype(np.float64)) - np.float64(mu)) / np.float64(sd)
    once, twice = bf16_bits(f, False), bf16_bits(f, True)
    silu = lambda v: bf16_bits(v / (1.0 + np.exp(-v.astype(np.float64))), False).astype(np.float64)
    pick = np.nonzero((once != twice) & (silu(once) != silu(twice)))[0]
    assert 5 <= pick.size < 200
    net = Mlp(S.N_FEAT, 256, 1, 1)
    W0, W1 = np.zeros((256, S.N_FEAT), np.float32), np.zeros((1, 256), np.float32)
    W0[0, 0] = W1[0, 0] = 1.0
    net.set_params(Mlp.flatten([(W0, np.zeros(256, np.float32)), (W1, np.zeros(1, np.float32))]))
    net.set_serving(MCS_FEATURES_SNOW_BRF, np.ones(1), np.zeros(1), np.zeros(1), S.FEAT_MU, S.FEAT_SD)
    x = S.sample_inputs(pick.size, 1).astype(np.float32)
    x[:, 0] = reff[pick]
    y = torch.empty(pick.size, 1, device='cuda')
    q = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    net.serve(q, pick.size, y)
    got = np.log(y[:, 0].cpu().numpy().astype(np.float64))
    net.close()
    # FP32 exponential: 1e-6 relative of a value below e^3, its logarithm 1e-6
    # absolute; one BF16 step of the smallest |feature| picked is far above
    want, wrong = silu(once[pick]), silu(twice[pick])
    assert np.abs(want - wrong).min() > 1e-5
    np.testing.assert_allclose(got, want, rtol=0, atol=5e-6)
