"""The event loops where they part: what a full cell leaves behind (addToCell,
EDMD.c:2576-2585, has no bound; the capacity is this library's), which loop a
batch gets (the reference has one, mainLoop, EDMD.c:5595-5630), and each of
them, deep calendars and windows of groups among them, against the oracle."""
import time

import numpy as np
import pytest

import edmd_fixtures as F
from test_gpu_wide import QUIET, VARIANTS, channel, same_state, same_trace

pytestmark = pytest.mark.gpu

FIELD = dict(wall_y=1, res_tan=1.0, add_field=1, field=-0.02)


@pytest.mark.parametrize("size,waves,res", [(1, 1, "RES_HBM"), (1, 1, "RES_LDS"),
                                            (2, 2, "RES_HBM"), (1100, 1, "RES_HBM")])
def test_state_after_a_full_cell(gpu, size, waves, res):
    """A crossing into a full cell stops the run with every disk's record as
    the events before it left them, on several wavefronts and on one."""
    st = F.lattice_state(200, 0.5, seed=3, lattice="fit")
    kw = dict(cell_capacity=4, trace_capacity=4000, **QUIET)

    def batch():
        b = gpu.Batch([st] * size, **kw)
        b.set_residency(getattr(gpu, res))
        b.set_loop_waves(waves)
        return b

    b = batch()
    with pytest.raises(gpu.EdmdError) as ei:
        b.run(max_events=4000)
    assert ei.value.code == 7
    o, after = b.observables(0), b.state(0)
    tr = b.trace(0)
    assert o["status"] == 7 and o["nevents"] == len(tr)
    assert tr["type"][-1] == gpu.EV_CELLCROSS and tr["i"][-1] == o["err_i"]
    c = batch()
    c.run(max_events=o["nevents"] - 1)
    same_state(after, c.state(0))
    same_trace(tr[:-1], c.trace(0))
    for k, v in b.events(0).items():
        np.testing.assert_array_equal(v, c.events(0)[k], err_msg=k)


def test_residency_names_the_loop_that_runs(gpu):
    """300 systems, two a compute unit: their arrays lie in LDS only where two
    of them fit it beside their windows (about 410 disks; one of 600 would)."""
    for n, lds in ((350, True), (450, False), (600, False)):
        st = F.lattice_state(n, 0.55, seed=n, lattice="fit")
        two = gpu.Batch([st] * 300)
        r = two.residency()
        assert r["lds"] == lds, (n, r)
        assert two.wavefronts() == (4 if n < 500 else 8)
        one = gpu.Batch([st])
        r1 = one.residency()
        assert r1["lds"] and one.wavefronts() == 8
        if lds:  # the wide loop's own: the arrays and the window
            assert r["lds_slots"] >= 300 and r["lds_bytes"] > n * 64 + 12 * n
        one.set_residency(gpu.RES_HBM)
        assert not one.residency()["lds"]
        rep = two.autotune(sweep_reps=0, trial_events=0)
        assert rep["in_lds"] == lds
        two.close()
        one.close()
    st = F.lattice_state(600, 0.55, seed=1, lattice="fit")
    b = gpu.Batch([st] * 300)
    b.set_loop_waves(2)
    assert b.wavefronts() == 1
    b.set_loop_waves(1)
    b.set_residency(gpu.RES_LDS)
    assert b.residency()["lds"]


def seconds(b, events, reps=3):
    """Median time of a run over so many more events of each system."""
    done, took = b.observables(0)["nevents"], []
    for _ in range(reps):
        done += events
        t = time.perf_counter()
        b.run(max_events=done)
        took.append(time.perf_counter() - t)
    return sorted(took)[reps // 2]


def test_any_cell_capacity_costs_alike(gpu):
    """The scan of cells that the LDS stage does not take (here 28 slots; 24
    are taken) reads one slot a candidate, not one cell after another, which
    took 2.4 times as long; both batches run on one wavefront a system."""
    st = F.lattice_state(200, 0.5, seed=3, lattice="fit")
    took = []
    for cap in (24, 28):
        b = gpu.Batch([st] * 1100, cell_capacity=cap)
        assert b.wavefronts() == 1
        b.run(max_events=500)
        took.append(seconds(b, 1000))
        b.close()
    assert took[1] < 1.6 * took[0], took


@pytest.mark.parametrize("n,phi,kw,size,waves", [
    (80, 0.5, {}, 1, 1), (100, 0.5, {}, 1, 4), (100, 0.5, {}, 300, 1), (128, 0.5, {}, 300, 4),
    (128, 0.5, dict(noise=2, dtnoise=0.1, temperature=1.0), 300, 1),
    (128, 0.5, {}, 1000, 1), (260, 0.5, {}, 1000, 4), (48, 0.2, {}, 1, 4),
    (160, 0.4, FIELD, 1, 1), (200, 0.4, FIELD, 1, 4), (200, 0.4, FIELD, 300, 1),
    (300, 0.4, FIELD, 300, 4), (16, 0.1, {}, 1, 1), (50, 0.5, dict(vr=0.3), 300, 1),
    (150, 0.5, dict(vr=0.3), 300, 4)])
def test_small_systems_take_one_wavefront(gpu, n, phi, kw, size, waves):
    """On either side of the cells that the loop of several wavefronts takes,
    by the systems that share a CU and by the reach of an event; the state of
    every copy is the same."""
    if "vr" in kw:
        st = gpu.init_random(n, phi, seed=n)
    else:
        st = F.lattice_state(n, phi, seed=n, lattice="fit")
    if "wall_y" in kw:
        st["y"] = 0.51 + st["y"] / st["Ly"] * (st["Ly"] - 1.02)
    b = gpu.Batch([st] * size, **kw)
    assert b.wavefronts() == waves
    b.run(max_events=3000, tmax=3.0 if "vr" in kw else 1e300)
    first = b.state(0)
    for k in range(1, size, 7):
        same_state(b.state(k), first)


@pytest.mark.parametrize("kw", [{}, FIELD, dict(noise=2, dtnoise=0.02, temperature=1.0)])
@pytest.mark.parametrize("n", [150, 1000, 6200])
def test_runs_of_any_length_match_oracle(gpu, oracle, n, kw):
    """Runs of a few events, which one wavefront handles, and of many, by
    events, collisions, time and kind, in turn on one system."""
    st = F.lattice_state(n, 0.4, seed=n, lattice="fit")
    if "wall_y" in kw:
        st["y"] = 0.51 + st["y"] / st["Ly"] * (st["Ly"] - 1.02)
    kw = dict(QUIET, **kw)
    s = gpu.System(st, trace_capacity=20000, **kw)
    done, seen = 0, []

    def after():
        seen.append(s.trace())
        return s.observables()

    for k in (1, 1, 7, 300, 10, 11, 2, 500, 1):
        done += k
        s.run(max_events=done)
        assert after()["nevents"] == done
    for k in (1, 2, 400, 3, 5):
        want = s.observables()["ncol"] + k
        s.run(max_collisions=want)
        assert after()["ncol"] == want
    for k in (1e-9, 1e-3, 0.05, 1e-4):
        t = s.observables()["t"] + k
        s.run(tmax=t)
        assert after()["t"] > t
    for kind in (gpu.EV_COLLISION, gpu.EV_CELLCROSS):
        s.run_until_kind(1 << kind)
        after()
        assert seen[-1]["type"][-1] == kind
    nev = s.observables()["nevents"]
    tr = np.concatenate(seen)
    assert len(tr) == nev
    o = oracle.Oracle(st, **kw)
    code, ref = o.run(nev)
    assert code == 0
    same_trace(tr, ref)
    same_state(s.state(), o.state())


def test_one_event_costs_alike_in_any_system(gpu):
    """A run of one event, of 2^18 disks and of 1000: the loop's window was
    read and its calendar made again for it, fifteen times as long."""
    took = []
    for n in (1000, 1 << 18):
        b = gpu.Batch([F.lattice_state(n, 0.4, seed=n, lattice="fit")])
        assert b.wavefronts() > 1
        b.run(max_events=2000)
        took.append(seconds(b, 1, reps=15))
        b.close()
    assert took[1] < 3 * took[0], took


def front(side):
    """Columns of a square grid closing on one another at one speed: half its
    collisions and crossings come at one time."""
    k = np.arange(side * side)
    L = side * 1.6
    return {"x": (k % side + 0.5) * (L / side), "y": (k // side + 0.5) * (L / side),
            "vx": np.where(k % 2 == 0, 1.0, -1.0), "vy": np.zeros(side * side),
            "rad": np.full(side * side, 0.5), "m": np.ones(side * side), "Lx": L, "Ly": L}


@pytest.mark.parametrize("side,waves", [(20, 8), (64, 16), (80, 16)])
def test_fronts_of_equal_times(gpu, side, waves):
    """Thousands of events at one time, more than a round's list takes, on
    several wavefronts and on one (windows of leaves and, at 6400 disks, of
    groups): the same events."""
    nev, got = 2 * side * side, []
    for cap in (0, 10):  # a capacity of 10 is the loop of one wavefront's
        b = gpu.Batch([front(side)], trace_capacity=nev, cell_capacity=cap, **QUIET)
        assert b.wavefronts() == (1 if cap else waves)
        b.run(max_events=nev)
        got.append((b.trace(0), b.state(0)))
        b.close()
    same_trace(got[0][0], got[1][0])
    same_state(got[0][1], got[1][1])


def test_lattice_start_costs_as_the_rest(gpu):
    """2000 disks on a square lattice, some on their cells' edges, which they
    cross at time 0: the first 8000 events took twice as long as the next."""
    st = gpu.init_lattice(2000, 0.3, seed=3)
    took = []
    for _ in range(3):
        b = gpu.Batch([st])
        took.append((seconds(b, 8000, reps=1), seconds(b, 8000, reps=1)))
        b.close()
    first, then = (min(t[k] for t in took) for k in (0, 1))
    assert first < 1.5 * then, took


def states_of(gpu, name, sizes):
    if "vr" in VARIANTS[name]:
        out = [gpu.init_random(n, 0.3, seed=n) for n in sizes]
        if "wall_x" in VARIANTS[name]:
            for st in out:
                for key in ("x", "y"):
                    st[key] = 0.51 + st[key] / st["Lx"] * (st["Lx"] - 1.02)
        return out
    if "wall_y" in VARIANTS[name]:
        return [channel(n, n) for n in sizes]
    return [F.lattice_state(n, 0.55, seed=n, lattice="fit") for n in sizes]


def batch_matches_oracle(gpu, oracle, name, sizes, copies, waves, nev, **engine):
    kw = dict(QUIET, **{k: v for k, v in VARIANTS[name].items() if "screen" not in k})
    base = states_of(gpu, name, sizes)
    b = gpu.Batch(base * copies, trace_capacity=nev, **kw, **engine)
    assert b.wavefronts() == waves
    b.run(max_events=nev // 3)
    b.run(max_events=nev)
    for k, st in enumerate(base):
        o = oracle.Oracle(st, **kw)
        code, tr = o.run(nev)
        assert code == 0
        at = (copies - 1) * len(base) + k
        same_trace(b.trace(at), tr)
        same_state(b.state(at), o.state())
    b.close()


@pytest.mark.parametrize("sizes,copies,waves", [((6400,), 1, 16), ((70, 70, 70, 6145), 1, 8),
                                                ((6200,), 260, 4)])
@pytest.mark.parametrize("name", ["plain", "thermostat", "walls", "field", "damping", "thermal",
                                  "grow", "grow_walls"])
def test_windows_of_groups_match_oracle(gpu, oracle, name, sizes, copies, waves):
    """Above 6144 disks the window is of groups of 64 leaves, of every system of
    the batch: on 16, 8 and 4 wavefronts."""
    batch_matches_oracle(gpu, oracle, name, sizes, copies, waves, 1500)


@pytest.mark.parametrize("name,n", [("plain", 262145), ("plain", 6400), ("walls", 6400),
                                    ("field", 6400), ("damping", 6400), ("thermal", 6400),
                                    ("grow", 6400), ("grow_walls", 6400), ("field", 262145),
                                    ("grow", 262145)])
def test_deep_calendars_on_one_wavefront_match_oracle(gpu, oracle, name, n):
    """The loop of one wavefront above 4096 disks (two levels of groups) and
    above 2^18 (three), which batches of more than four systems a compute unit
    run; here by a cell capacity that the other loop does not take."""
    batch_matches_oracle(gpu, oracle, name, (n,), 1, 1, 1500, cell_capacity=30)


@pytest.mark.parametrize("name", list(VARIANTS))
def test_four_and_eight_wavefronts_agree_with_one(gpu, name):
    """Three systems of 350 to 400 disks alone (8 wavefronts each, arrays in
    LDS), in batches of 300 and 600 (4) and of 1200 (1): states, counters, sums,
    thermo rows and calendars alike."""
    base = states_of(gpu, name, (350, 380, 400))
    got = []
    for size, waves in ((1200, 1), (3, 8), (300, 4), (600, 4)):
        b = gpu.Batch(base * (size // 3), **VARIANTS[name])
        assert b.wavefronts() == waves, size
        b.run(max_events=1500)
        b.run(max_events=4000, tmax=12.0)
        got.append([(b.state(size - 3 + k), b.observables(size - 3 + k), b.thermo(size - 3 + k),
                     b.calendar(size - 3 + k)) for k in range(3)])
        b.close()
    for other in got[1:]:
        for (sa, oa, ta, ca), (sb, ob, tb, cb) in zip(got[0], other):
            same_state(sb, sa)
            assert oa == ob
            assert np.array_equal(ta.view(np.uint8), tb.view(np.uint8))
            for k in ca:
                assert np.array_equal(np.asarray(ca[k]).view(np.uint8),
                                      np.asarray(cb[k]).view(np.uint8)), k


@pytest.mark.parametrize("n,mode,res", [(300, "run", "RES_AUTO"), (400, "run", "RES_AUTO"),
                                        (900, "run", "RES_AUTO"), (50, "grow", "RES_AUTO"),
                                        (300, "grow", "RES_AUTO"), (300, "grow", "RES_HBM")])
def test_copies_that_share_a_compute_unit_end_alike(gpu, n, mode, res):
    """512 copies, two a compute unit: each ends as the one alone does."""
    if mode == "run":
        st, kw, run = F.lattice_state(n, 0.6, seed=n, lattice="fit"), {}, dict(max_events=12000)
    else:
        st, kw, run = gpu.init_random(n, 0.55, seed=n), dict(vr=0.3), dict(max_events=30000, tmax=2.0)
    ends = []
    for size in (1, 512):
        b = gpu.Batch([st] * size, **kw)
        b.set_residency(getattr(gpu, res))
        b.run(**run)
        ends.append([b.state(k) for k in range(size)])
        b.close()
    for s in ends[1]:
        same_state(s, ends[0][0])
