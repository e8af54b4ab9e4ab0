"""g(r) by sorted positions and culled tiles against the oracle's loop over
all pairs (calculate_pcf, pcf.c:16-75): both sides of the rule that sorts
(4096 disks, the range of distances against the box), ragged tiles, positions
outside the box and not a number, one bin and the most there can be.  Counts
are whole numbers: equal to the last bit."""
import numpy as np
import pytest

import edmd_fixtures as F

pytestmark = pytest.mark.gpu


def bits(a):
    return np.asarray(a, np.float64).view(np.uint64)


def positions(n, Lx, Ly, seed, out=False):
    r = np.random.default_rng(seed)
    x, y = r.random(n) * Lx, r.random(n) * Ly
    if out:
        x[::7] += Lx * r.integers(-2, 3, len(x[::7]))
        y[::11] -= 1.4 * Ly
        x[n // 3] = np.nan
        y[n // 2] = np.inf
        x[5:9] = x[4]
        y[5:9] = y[4]
    return x, y


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 4095, 4096, 4097, 9001])
@pytest.mark.parametrize("out", [False, True])
def test_pcf_both_sides_of_the_sort(gpu, oracle, n, out):
    if out and n < 63:
        pytest.skip("no room for the odd positions")
    Lx, Ly = 70.0, 41.0
    x, y = positions(n, Lx, Ly, n, out)
    for dr, max_r in ((0.05, 5.0), (0.1, 20.5), (0.3, 60.0)):
        r0, g0 = oracle.pcf(x, y, Lx, Ly, dr, max_r)
        r1, g1 = gpu.pcf(x, y, Lx, Ly, dr, max_r)
        assert np.array_equal(bits(r0), bits(r1))
        assert np.array_equal(bits(g0), bits(g1)), (n, dr, max_r)


@pytest.mark.parametrize("bins", [1, 32768])
def test_pcf_bins(gpu, oracle, bins):
    x, y = positions(5000, 50.0, 60.0, bins)
    dr = 4.0 / bins  # a power of two: max_r / dr is the number of bins
    r0, g0 = oracle.pcf(x, y, 50.0, 60.0, dr, 4.0)
    r1, g1 = gpu.pcf(x, y, 50.0, 60.0, dr, 4.0)
    assert len(g1) == bins and np.array_equal(bits(g0), bits(g1))


def test_pcf_distances_on_the_edges(gpu, oracle):
    """A lattice whose distances are whole numbers of bins."""
    k = np.arange(70)
    x, y = (a.ravel().astype(float) for a in np.meshgrid(k, k))
    for dr in (0.5, 0.1):
        r0, g0 = oracle.pcf(x, y, 70.0, 70.0, dr, 10.0)
        r1, g1 = gpu.pcf(x, y, 70.0, 70.0, dr, 10.0)
        assert np.array_equal(bits(g0), bits(g1))


def test_pcf_of_a_batch_flown_to_its_time(gpu, oracle):
    st = F.lattice_state(4900, 0.5, seed=3, lattice="fit")
    b = gpu.Batch([st])
    b.run(max_events=20000)
    r1, g1 = b.pcf(0, 0.05, 6.0, extrapolate=True)
    o = oracle.Oracle(st)
    o.run(20000, trace=False)
    o.sync_all(b.observables(0)["t"])
    s = o.state()
    r0, g0 = oracle.pcf(s["x"], s["y"], st["Lx"], st["Ly"], 0.05, 6.0)
    assert np.array_equal(bits(g0), bits(g1))
