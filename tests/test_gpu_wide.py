"""The event loop of one system on a workgroup of several wavefronts against
the oracle and against the loop of one wavefront, bit for bit.

Small disk counts here run four wavefronts a system in batches of up to four
systems per compute unit; the other widths, and those batches against the loop
of one wavefront, are in test_gpu_wide_widths.py.  The results may not depend
on it.  The reference runs one event at a time
(mainLoop, EDMD.c:5595-5630)."""
import numpy as np
import pytest

import edmd_fixtures as F
from conftest import bits

pytestmark = pytest.mark.gpu

QUIET = dict(first_screen=1e9, dtime=1e9, first_thermo=1e9)


def same_trace(got, ref):
    assert len(got) == len(ref)
    for k in ("type", "i", "j", "valid"):
        bad = np.nonzero(got[k] != ref[k])[0]
        assert len(bad) == 0, "%s differs first at event %d" % (k, bad[0])
    np.testing.assert_array_equal(bits(got["t"]), bits(ref["t"]))


def same_state(got, ref):
    for k in ("x", "y", "vx", "vy", "t"):
        np.testing.assert_array_equal(bits(got[k]), bits(ref[k]), err_msg=k)
    for k in ("coll", "cx", "cy"):
        np.testing.assert_array_equal(np.asarray(got[k], dtype=np.int64),
                                      np.asarray(ref[k], dtype=np.int64), err_msg=k)


def against_oracle(gpu, oracle, st, nev, kw, **engine):
    s = gpu.System(st, trace_capacity=nev, **kw, **engine)
    # in two runs: the second starts from the calendar the first wrote back
    s.run(max_events=nev // 3)
    s.run(max_events=nev)
    o = oracle.Oracle(st, **kw)
    code, tr = o.run(nev)
    assert code == 0
    same_trace(s.trace(), tr)
    same_state(s.state(), o.state())
    a, b = s.observables(), o.observables()
    for k in ("ncol", "ncross"):
        assert a[k] == b[k]


# the window's levels: leaves (up to 6144 disks), groups of 64 leaves (up to
# 262144), groups of 4096; and the smallest systems (five cells a side: the
# reference ends in an overlap in much smaller boxes)
@pytest.mark.parametrize("n,phi", [(2, 0.012), (3, 0.02), (64, 0.5), (65, 0.6), (6144, 0.6),
                                   (6145, 0.65), (262144, 0.5), (262145, 0.5)])
def test_window_levels_match_oracle(gpu, oracle, n, phi):
    st = F.lattice_state(n, phi, seed=n, lattice="fit")
    against_oracle(gpu, oracle, st, 3000, QUIET)


@pytest.mark.parametrize("cap", [10, 24, 28])
def test_cell_capacities_match_oracle(gpu, oracle, cap):
    """Capacities the staged scan takes (24) and does not (rows that are not
    whole 16-byte chunks, more than 24 slots)."""
    st = F.lattice_state(500, 0.6, seed=cap, lattice="fit")
    against_oracle(gpu, oracle, st, 6000, QUIET, cell_capacity=cap)


def test_equal_times_agree(gpu):
    """Columns of a square grid closing on one another at one speed: hundreds
    of collisions and crossings at exactly equal times, more than a round
    takes; in batches of 1, 300 and 600."""
    side = 20
    k = np.arange(side * side)
    L = 32.0
    st = {"x": (k % side + 0.5) * (L / side), "y": (k // side + 0.5) * (L / side),
          "vx": np.where(k % 2 == 0, 1.0, -1.0), "vy": np.zeros(side * side),
          "rad": np.full(side * side, 0.5), "m": np.ones(side * side), "Lx": L, "Ly": L}
    got = []
    for size in (1, 300, 600):
        b = gpu.Batch([st] * size, trace_capacity=4000, **QUIET)
        b.set_residency(gpu.RES_HBM)
        b.run(max_events=4000)
        got.append((b.trace(size - 1), b.state(size - 1)))
        b.close()
    for tr, state in got[1:]:
        same_trace(tr, got[0][0])
        same_state(state, got[0][1])


def channel(n, seed):
    st = F.lattice_state(n, 0.4, seed=seed, lattice="fit")
    for key in ("x", "y"):
        st[key] = 0.51 + st[key] / st["Lx"] * (st["Lx"] - 1.02)
    return st


VARIANTS = {
    "plain": dict(first_thermo=0.2, dtime_thermo=0.2, first_screen=0.3, dtime=0.3),
    "thermostat": dict(noise=2, dtnoise=0.15, temperature=1.3),
    "walls": dict(wall_x=1, wall_y=1, res_wall=0.9, res_tan=0.5, first_thermo=0.2,
                  dtime_thermo=0.2),
    "field": dict(wall_y=1, res_tan=1.0, add_field=1, field=-0.05),
    "damping": dict(damping=1, gamma=0.05),
    "thermal": dict(wall_x=1, wall_y=1, thermal_wall=1, temperature=0.8, rng_seed=7),
    "grow": dict(vr=0.3),
    "grow_walls": dict(vr=0.3, wall_x=1, wall_y=1),
}


@pytest.mark.parametrize("name", list(VARIANTS))
def test_loop_widths_agree(gpu, name):
    """The same systems in batches of 3, 300 and 600: states, counters, sums and thermo rows alike."""
    kw = VARIANTS[name]
    if "vr" in kw:
        base = [gpu.init_random(n, 0.4, seed=n) for n in (70, 120, 200)]
        if "wall_x" in kw:
            for st in base:
                for key in ("x", "y"):
                    st[key] = 0.51 + st[key] / st["Lx"] * (st["Lx"] - 1.02)
    elif "wall_y" in kw:
        base = [channel(n, n) for n in (70, 120, 200)]
    else:
        base = [F.lattice_state(n, 0.55, seed=n, lattice="fit") for n in (70, 120, 200)]
    got = []
    for size in (3, 300, 600):
        b = gpu.Batch(base * (size // 3), **kw)
        b.set_residency(gpu.RES_HBM)
        b.run(max_events=1500)
        b.run(max_events=4000, tmax=12.0)
        at = size - 3
        got.append([(b.state(at + k), b.observables(at + k), b.thermo(at + k), b.calendar(at + k))
                    for k in range(3)])
        b.close()
    for other in got[1:]:
        for (sa, oa, ta, ca), (sb, ob, tb, cb) in zip(got[0], other):
            same_state(sb, sa)
            assert oa == ob
            assert np.array_equal(ta.view(np.uint8), tb.view(np.uint8))
            for k in ca:
                assert np.array_equal(np.asarray(ca[k]).view(np.uint8),
                                      np.asarray(cb[k]).view(np.uint8)), k
