"""Walks whose photons fit in the launch's lanes run one chunk per block (no
queue); larger ones the chunk queue.  Both give the records of every photon
bit for bit (coop_live 0, polarised and replay walks), at the sizes around the
line between them, for one and for several cases, into the context's buffers
and into a caller's."""
import numpy as np
import pytest

from tests.golden_cases import load
from tests.gpu_cases import case_from_params
from tests.test_gpu_native import gpu_case
from tests.test_oracle_golden import META, run_case

pytestmark = pytest.mark.gpu
FIELDS = ('condition', 'band', 'n_scat', 'theta_n', 'phi_n', 'path_length', 'wvn')
QUEUE = (64, 1, 64, 4, 0)        # 64 lanes per CU: anything above 64 x CUs photons goes through the queue


@pytest.fixture(scope='module')
def walker():
    from monte_carlompi_amd.gpu import GpuWalker
    w = GpuWalker(0)
    yield w
    w.close()


def records(walker, shape, cases, stokes=False, **kw):
    walker.set_cases(cases)
    walker.set_launch(*shape)
    walker.walk(seed=77, records=True, **kw)
    r = walker.records()
    if stokes:
        r.update(walker.stokes())
    return r, walker.counts(), walker.tallies()


def assert_same(a, b, fields=FIELDS):
    for f in fields:
        np.testing.assert_array_equal(a[0][f], b[0][f], err_msg=f)
    np.testing.assert_array_equal(a[1], b[1])
    np.testing.assert_allclose(a[2], b[2], rtol=1e-12, atol=1e-9)   # FP64 sums in another order


@pytest.mark.parametrize('n', [1, 63, 1025, 20_011, 262_143, 262_144, 262_145, 300_001])
def test_one_chunk_per_block_gives_the_queue_records(walker, n):
    case = gpu_case(n, 20.0, 30.0, True, 0.5, g=0.87, ssa=0.995)
    ref = records(walker, QUEUE, [case])
    assert int(ref[1][0, 0]) == n
    for shape in [(256, 4, 2048, 8, 0), (1024, 1, 1954, 16, 0), (256, 6, 8192, 16, 0), (256, 5, 300, 8, 0)]:
        assert_same(records(walker, shape, [case]), ref)


def test_several_cases(walker):
    """Uneven cases, one of them empty, their chunks never shared."""
    cases = [gpu_case(n, 8.0 + k, 10.0 * k, k % 2 == 0, 0.4, g=0.8, ssa=0.99)
             for k, n in enumerate([1, 5000, 2, 313, 12_001, 64])]
    cases[2].n_photons = 0
    ref = records(walker, (64, 1, 64, 4, 0), cases)
    for shape in [(256, 4, 2048, 8, 0), (512, 2, 2048, 8, 0)]:
        assert_same(records(walker, shape, cases), ref)
    many = [gpu_case(n, 5.0, 20.0, False, 0.0, g=0.8, ssa=0.95) for n in range(1, 300)]
    ref = records(walker, QUEUE, many)
    assert_same(records(walker, (256, 4, 2048, 8, 0), many), ref)


@pytest.mark.parametrize('n', [1, 1500, 131_073, 196_609])
def test_polar(walker, tmp_path, n):
    from monte_carlompi_amd.workloads import snow_polar_case
    case = snow_polar_case(n, str(tmp_path))
    ref = records(walker, QUEUE, [case], stokes=True)
    for shape in [(256, 4, 2048, 8, 16), (512, 2, 1024, 16, 0), (256, 3, 1302, 16, 16)]:
        assert_same(records(walker, shape, [case], stokes=True), ref, FIELDS + ('Q_n', 'U_n', 'V_n'))


@pytest.mark.parametrize('name', [c['name'] for c in load()[1] if not c['lowprec_columns']])
def test_replay_chunks(walker, name):
    """The queue and the ONE form, with the tail that builds a photon's next
    steps in the idle lanes, on the reference's own streams (Lambertian bottoms
    and surfaces among them)."""
    golden = [c for c in load()[1] if c['name'] == name][0]
    _, par, values, offsets = run_case(golden)
    k = 64 * walker.cus // golden['n'] + 2                 # past the queue shape's lanes
    case, band = case_from_params(par, golden['tau'], META['rho_snw'], golden['theta0'], golden['lb'], golden['R'],
                                  golden.get('ls', False))
    case.n_photons = k * golden['n']
    off = np.concatenate([[0], (offsets[-1] * np.arange(k)[:, None] + offsets[1:][None, :]).ravel()])
    kw = dict(mode='replay', replay=(np.tile(values, k), off), photon_band=np.tile(band, k))
    a = records(walker, QUEUE, [case], **kw)
    b = records(walker, (256, 4, 512, 8, 0), [case], **kw)
    assert_same(a, b)
    np.testing.assert_array_equal(a[0]['n_scat'], np.tile(golden['records']['n_scat'], k))


def test_caller_buffers(walker):
    import torch
    n = 20_011
    case = gpu_case(n, 20.0, 30.0, True, 0.5, g=0.87, ssa=0.995)
    ref = records(walker, QUEUE, [case])
    walker.set_launch(256, 4, 2048, 8, 0)
    dev = dict(device='cuda')
    tal = torch.zeros(1, 656, dtype=torch.float64, **dev)
    cnt = torch.zeros(1, 16, dtype=torch.int64, **dev)
    rec = {k: torch.zeros(n, dtype=torch.int32 if k in ('n_scat', 'cond_band') else torch.float32, **dev)
           for k in ('n_scat', 'cond_band', 'theta_n', 'phi_n', 'path_length')}
    torch.cuda.synchronize()
    walker.walk_noalloc(tal, cnt, records=rec, seed=77)
    np.testing.assert_array_equal(rec['n_scat'].cpu().numpy(), ref[0]['n_scat'])
    np.testing.assert_array_equal((rec['cond_band'] & 0xff).cpu().numpy(), ref[0]['condition'])
    np.testing.assert_array_equal(rec['theta_n'].double().cpu().numpy(), ref[0]['theta_n'])
    np.testing.assert_array_equal(cnt.cpu().numpy().astype(np.uint64), ref[1])


@pytest.mark.parametrize('n', [3, 5_003, 65_536])
def test_small_cooperative_walks_keep_the_law(walker, n):
    """Default mode, every wave in the cooperative tail from its first step:
    condition fractions against the one-lane walk's."""
    from tests.test_gpu_native import two_sample_z
    case = gpu_case(n, 20.0, 30.0, True, 0.5, g=0.87, ssa=0.995)
    walker.set_cases([case])
    got = {}
    for coop in (16, 0):
        walker.set_launch(256, 4, 2048, 8, coop)
        k = np.zeros(16, np.uint64)
        for s in range(4):
            walker.walk(seed=500 + 10 * coop + s, records=True)
            k += walker.counts()[0]
            assert int(np.sum(walker.records()['n_scat'] + 1)) == int(walker.counts()[0, 8])
        got[coop] = k
    assert int(got[16][0]) == 4 * n
    assert n < 100 or float(got[16][9]) > 0.9 * float(got[16][8])
    for cond in (1, 2, 4):
        assert abs(two_sample_z(int(got[16][cond]), 4 * n, int(got[0][cond]), 4 * n)) < 4
