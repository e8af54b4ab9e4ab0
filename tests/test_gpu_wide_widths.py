"""The event loop on 16, 8 and 4 wavefronts a system against the loop of one
wavefront, bit for bit, at the disk counts and batch sizes where its width
changes; and a batch whose systems have different window levels against the
oracle.  The reference runs one event at a time (mainLoop, EDMD.c:5595-5630).
"""
import numpy as np
import pytest

import edmd_fixtures as F
from test_gpu_wide import QUIET, VARIANTS, channel, same_state, same_trace

pytestmark = pytest.mark.gpu


def systems(gpu, name, sizes):
    kw = VARIANTS[name]
    if "vr" in kw:
        out = [gpu.init_random(n, 0.35, seed=n) for n in sizes]
        if "wall_x" in kw:
            for st in out:
                for key in ("x", "y"):
                    st[key] = 0.51 + st[key] / st["Lx"] * (st["Lx"] - 1.02)
        return out
    if "wall_y" in kw:
        return [channel(n, n) for n in sizes]
    return [F.lattice_state(n, 0.55, seed=n, lattice="fit") for n in sizes]


@pytest.mark.parametrize("name", list(VARIANTS))
def test_sixteen_wavefronts_agree(gpu, name):
    """Batches of 3 (16 wavefronts a system), 300 (8), 600 (4) and 1200 (1)."""
    base = systems(gpu, name, (1700, 1850, 2000))
    got = []
    for size in (3, 300, 600, 1200):
        b = gpu.Batch(base * (size // 3), **VARIANTS[name])
        b.set_residency(gpu.RES_HBM)
        b.run(max_events=900)
        b.run(max_events=3000)
        at = size - 3
        got.append([(b.state(at + k), b.observables(at + k), b.thermo(at + k), b.calendar(at + k))
                    for k in range(3)])
        b.close()
    for other in got[:-1]:
        for (sa, oa, ta, ca), (sb, ob, tb, cb) in zip(got[-1], other):
            same_state(sb, sa)
            assert oa == ob
            assert np.array_equal(ta.view(np.uint8), tb.view(np.uint8))
            for k in ca:
                assert np.array_equal(np.asarray(ca[k]).view(np.uint8),
                                      np.asarray(cb[k]).view(np.uint8)), k


@pytest.mark.parametrize("sizes", [(299,), (300,), (1799,), (1800,), (300, 6200, 2000),
                                   (70, 6145)])
def test_widths_and_mixed_levels_match_oracle(gpu, oracle, sizes):
    nev = 4000
    base = [F.lattice_state(n, 0.6, seed=n, lattice="fit") for n in sizes]
    b = gpu.Batch(base, trace_capacity=nev, **QUIET)
    b.run(max_events=nev // 3)
    b.run(max_events=nev)
    for k, st in enumerate(base):
        o = oracle.Oracle(st, **QUIET)
        code, tr = o.run(nev)
        assert code == 0
        same_trace(b.trace(k), tr)
        same_state(b.state(k), o.state())


@pytest.mark.parametrize("n", [16, 17])
def test_equal_times_in_wide_rounds(gpu, n):
    """Pairs far apart that collide at exactly equal times: more of them than
    a round of 16 takes, on 16 wavefronts and on one."""
    pairs = 1000
    side = 32
    k = np.arange(2 * pairs)
    L = side * 6.0
    col, row = (k // 2) % side, (k // 2) // side
    st = {"x": col * 6.0 + 1.5 + (k % 2) * 2.0, "y": row * 6.0 + 1.5 + (n % 2) * 0.01,
          "vx": np.where(k % 2 == 0, 1.0, -1.0), "vy": np.zeros(2 * pairs),
          "rad": np.full(2 * pairs, 0.5), "m": np.ones(2 * pairs), "Lx": L, "Ly": L}
    got = []
    for size in (1, 1200):
        b = gpu.Batch([st] * size, trace_capacity=3000, **QUIET)
        b.set_residency(gpu.RES_HBM)
        b.run(max_events=3000)
        got.append((b.trace(size - 1), b.state(size - 1)))
        b.close()
    same_trace(got[1][0], got[0][0])
    same_state(got[1][1], got[0][1])


@pytest.mark.parametrize("n", [350, 400, 430])
@pytest.mark.parametrize("name", ["plain", "thermostat", "grow", "walls"])
def test_two_systems_a_unit_in_lds_agree(gpu, name, n):
    """300 systems, two a compute unit, with their arrays in LDS where two of
    them fit it beside their windows (about 410 disks) and in HBM above that;
    against the loop of one wavefront (1200)."""
    base = systems(gpu, name, (n, n - 1, n - 50))
    got = []
    for size in (300, 1200):
        b = gpu.Batch(base * (size // 3), **VARIANTS[name])
        b.set_residency(gpu.RES_AUTO if size == 300 else gpu.RES_HBM)
        b.run(max_events=900)
        b.run(max_events=3000)
        at = size - 3
        got.append([(b.state(at + k), b.observables(at + k), b.thermo(at + k), b.calendar(at + k))
                    for k in range(3)])
        b.close()
    for (sa, oa, ta, ca), (sb, ob, tb, cb) in zip(*got):
        same_state(sa, sb)
        assert oa == ob
        assert np.array_equal(ta.view(np.uint8), tb.view(np.uint8))
        for k in ca:
            assert np.array_equal(np.asarray(ca[k]).view(np.uint8),
                                  np.asarray(cb[k]).view(np.uint8)), k
