"""Walks dealt out once over the chip against the chunk queue, with the queue's
records taken from a walk of more photons than fit the other form: a photon's
walk is a function of (seed, case, photon) alone, so the first n records of the
large walk are those of n photons walked by themselves, bit for bit.

A walk has a lane for every photon up to 1,024 photons per CU (coop_live 0), a
polarised one up to 768: 512-thread blocks, one per CU, up to 512 and
256-thread blocks above."""
import numpy as np
import pytest

from tests.test_gpu_native import gpu_case

pytestmark = pytest.mark.gpu
FIELDS = ('condition', 'band', 'n_scat', 'theta_n', 'phi_n', 'path_length', 'wvn')
STOKES = ('Q_n', 'U_n', 'V_n')
SEED = 4711


@pytest.fixture(scope='module')
def walker():
    from monte_carlompi_amd.gpu import GpuWalker
    w = GpuWalker(0)
    yield w
    w.close()


def walk(walker, shape, case, n, stokes=False, graph=False):
    case.n_photons = n
    walker.set_cases([case])
    walker.set_launch(*shape)
    walker.walk(seed=SEED, records=True, use_graph=graph)
    r = walker.records()
    if stokes:
        r.update(walker.stokes())
    assert int(walker.counts()[0, 0]) == n
    return r


def assert_first(ref, got, n, fields, what):
    for f in fields:
        np.testing.assert_array_equal(got[f], ref[f][:n], err_msg='%s %s' % (what, f))


@pytest.fixture(scope='module')
def hg(walker):
    """300,001 photons or 1,024 per CU and more, one lane to the end of each walk: no tail mode."""
    case = gpu_case(1, 20.0, 30.0, True, 0.5, g=0.87, ssa=0.995)
    n = max(300_001, 1024 * walker.cus + 37_857)
    return case, n, walk(walker, (256, 6, 8192, 16, 0), case, n)


@pytest.mark.parametrize('shape', [(256, 4, 2048, 8, 0), (1024, 1, 4096, 64, 0), (512, 2, 8192, 32, 0), (64, 8, 64, 1, 0),
                                   (256, 5, 2048, 8, 0), (256, 6, 1024, 8, 0)])
def test_queue_instances_eager_and_through_graphs(walker, hg, shape):
    """Every register budget's queue instance, with the packet tail (up to four
    waves per SIMD) and without, launched and replayed."""
    case, n, ref = hg
    assert_first(ref, walk(walker, shape, case, n), n, FIELDS, shape)
    for _ in range(3):
        assert_first(ref, walk(walker, shape, case, n, graph=True), n, FIELDS, (shape, 'graph'))


@pytest.mark.parametrize('per_cu', [None, 5, 256, 1000, 1024])
@pytest.mark.parametrize('shape', [(256, 4, 2048, 8, 0), (1024, 1, 1954, 16, 0), (256, 6, 8192, 16, 0)])
def test_dealt_out_once(walker, hg, shape, per_cu):
    case, _, ref = hg
    for n in [1, 63, 1025] if per_cu is None else [per_cu * walker.cus, per_cu * walker.cus - 65]:
        assert_first(ref, walk(walker, shape, case, n), n, FIELDS, (shape, n))


@pytest.fixture(scope='module')
def polar(walker, tmp_path_factory):
    """Polarised photons past the other form, without the tail mode."""
    from monte_carlompi_amd.workloads import snow_polar_case
    case = snow_polar_case(1, str(tmp_path_factory.mktemp('tables')))
    n = 768 * walker.cus + 3_395
    return case, n, walk(walker, (512, 2, 2048, 16, 0), case, n, stokes=True)


@pytest.mark.parametrize('shape', [(512, 2, 2048, 16, 16), (256, 4, 1024, 8, 8), (1024, 1, 600, 16, 16),
                                   (384, 2, 1024, 16, 16), (256, 3, 1302, 16, 16), (128, 4, 512, 8, 0)])
def test_polar_queue_and_tail(walker, polar, shape):
    case, n, ref = polar
    assert_first(ref, walk(walker, shape, case, n, stokes=True), n, FIELDS + STOKES, shape)
    assert_first(ref, walk(walker, shape, case, n, stokes=True, graph=True), n, FIELDS + STOKES, (shape, 'graph'))


@pytest.mark.parametrize('coop', [0, 16])
@pytest.mark.parametrize('per_cu,less', [(0, -1), (0, -1500), (5, 3), (512, 0), (512, -1), (700, 9), (768, 0)])
def test_polar_dealt_out_once(walker, polar, per_cu, less, coop):
    """Both block sizes of the form, at their edges, with and without tail."""
    case, _, ref = polar
    n = per_cu * walker.cus - less
    assert_first(ref, walk(walker, (256, 4, 2048, 8, coop), case, n, stokes=True), n, FIELDS + STOKES, (n, coop))


@pytest.mark.parametrize('per_cu', [100, 600])
def test_polar_dealt_out_once_into_caller_memory(walker, polar, per_cu):
    import torch
    case, _, ref = polar
    n = case.n_photons = per_cu * walker.cus + 1
    walker.set_cases([case])
    walker.set_launch(256, 4, 2048, 8, 16)
    tal = torch.zeros(1, 656, dtype=torch.float64, device='cuda')
    cnt = torch.zeros(1, 16, dtype=torch.int64, device='cuda')
    rec = {k: torch.zeros(n, dtype=torch.int32 if k in ('n_scat', 'cond_band') else torch.float32, device='cuda')
           for k in ('n_scat', 'cond_band', 'theta_n', 'phi_n', 'path_length')}
    st = torch.zeros(3, n, dtype=torch.float32, device='cuda')
    torch.cuda.synchronize()
    walker.walk_noalloc(tal, cnt, records=rec, stokes=st, seed=SEED)
    np.testing.assert_array_equal(rec['n_scat'].cpu().numpy(), ref['n_scat'][:n])
    np.testing.assert_array_equal((rec['cond_band'] & 0xff).cpu().numpy(), ref['condition'][:n])
    for f in ('theta_n', 'phi_n', 'path_length'):
        np.testing.assert_array_equal(rec[f].double().cpu().numpy(), ref[f][:n], err_msg=f)
    for k, f in enumerate(STOKES):
        np.testing.assert_array_equal(st[k].double().cpu().numpy(), ref[f][:n], err_msg=f)
    assert int(cnt[0, 0]) == n
