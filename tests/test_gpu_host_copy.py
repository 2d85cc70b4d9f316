"""Large copies between the device and pageable host arrays (the pinned ring
and its host threads) move the same bytes as the runtime's own copies."""
import numpy as np
import pytest

from tests.gpu_cases import case_from_params
from tests.test_gpu_native import EXT100

pytestmark = pytest.mark.gpu
N_OUT = 651
SLOT = (2 << 20) / (4 * N_OUT)      # rows of one 2 MB slot


@pytest.fixture(scope='module')
def net():
    from monte_carlompi_amd.mlp import Mlp
    m = Mlp(5, 256, 2, N_OUT, max_batch=16384)
    m.set_params(np.random.default_rng(3).normal(0.0, 0.1, m.n_params).astype(np.float32))
    yield m
    m.close()


@pytest.mark.parametrize('n', [int(4 * SLOT), int(4 * SLOT) + 1, int(5 * SLOT) + 1, int(9 * SLOT) + 3, 16384, 16385,
                               40_007])
def test_forward_rows(net, n):
    """Output columns of n rows against the same rows in calls small enough
    for the runtime's copy: equal bit for bit (each row is independent)."""
    x = np.random.default_rng(n).normal(0.0, 1.0, (n, 5)).astype(np.float32)
    y = net.forward(x)
    ref = np.concatenate([net.forward(x[a:a + 1024]) for a in range(0, n, 1024)])
    np.testing.assert_array_equal(y, ref)


@pytest.mark.parametrize('n', [1, 9600, 20_011])
def test_replay_upload(n):
    """A recorded stream from a pageable array (the ring from 16 MB) and from
    pinned memory (one DMA): the same records."""
    import torch
    from monte_carlompi_amd.gpu import GpuWalker
    from oracle import coracle
    ext = EXT100 * 300.0

    def ssp(wvls):
        k = wvls.size
        return (dict(ssa=np.full(k, 0.99), ext=np.full(k, EXT100), g=np.full(k, 0.89)),
                dict(ssa=np.zeros(k), ext=np.zeros(k)))
    out, par = coracle.run_rank(7, n, 1.3, 1e-12, ssp, 0.0, ext, 300.0, 60.0, True, 0.5, record=True)
    values, offsets = out['stream']
    case, band = case_from_params(par, ext, 300.0, 60.0, True, 0.5)
    pinned = torch.from_numpy(values).pin_memory()
    w = GpuWalker(0)
    try:
        w.set_cases([case])
        got = []
        for v in (values, pinned.numpy()):
            w.walk(mode='replay', replay=(v, offsets), photon_band=band, records=True)
            got.append(w.records())
        for k in got[0]:
            np.testing.assert_array_equal(got[0][k], got[1][k], err_msg=k)
        np.testing.assert_array_equal(got[0]['n_scat'], out['n_scat'])
        np.testing.assert_array_equal(got[0]['condition'], out['condition'])
    finally:
        w.close()
