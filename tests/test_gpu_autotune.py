"""mcs_autotune with a photon cap times the candidates as they would run on the
whole walk.  The cap leaves few enough photons that a walk of them alone would
be dealt out once over the chip, with the same launch whatever the candidate."""
import pytest

from tests.test_gpu_native import gpu_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def walker():
    from monte_carlompi_amd.gpu import GpuWalker
    w = GpuWalker(0)
    yield w
    w.close()


@pytest.mark.parametrize('kind', ['polar', 'reproducible'])
def test_capped_candidates_differ(walker, tmp_path, kind):
    """40,000 photons in chunks of 256 (157 blocks) and of 8,192 (5 blocks of 256
    threads, 32 rounds of photons through each lane), as a walk of 8.4e6 takes them
    (below 8,192 photons a block of the grid the larger chunks would shrink)."""
    from monte_carlompi_amd.workloads import snow_polar_case
    n = 8_192 * 4 * walker.cus
    case = snow_polar_case(n, str(tmp_path)) if kind == 'polar' else gpu_case(n, 20.0, 30.0, True, 0.5, g=0.87, ssa=0.995)
    walker.set_cases([case])
    coop = 16 if kind == 'polar' else 0
    few, many = (256, 3, 8192, 16, coop), (256, 3, 256, 16, coop)
    best, times = walker.autotune([few, many], photons_cap=40_000, repeats=3)
    print(kind, 'ms', list(times), flush=True)
    assert times[0] > 1.5 * times[1]
    assert tuple(best) == many
    # the walk afterwards is the whole one
    walker.walk(seed=1, records=False)
    assert int(walker.counts()[0, 0]) == n


def test_cap_above_the_cases_changes_nothing(walker):
    """With nothing cut off, a small walk is timed as it runs (dealt out once):
    both candidates are then one launch."""
    walker.set_cases([gpu_case(20_000, 20.0, 30.0, True, 0.5, g=0.87, ssa=0.995)])
    best, times = walker.autotune([(256, 4, 8192, 16, 0), (256, 4, 256, 16, 0)], photons_cap=40_000, repeats=5)
    assert abs(times[0] - times[1]) < 0.3 * times[1]
