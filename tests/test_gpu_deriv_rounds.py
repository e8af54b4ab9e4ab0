"""Tangent and adjoint passes where their chunks of 64 records can go wrong:
tapes of none, one and about one or two chunks, few disks (every record of a
chunk waits for others), more disks than the chunk's table has slots, and
vectors in HBM; walls among the records.  Bit for bit the oracle's, which
applies one record after another.
"""
import ctypes as C

import numpy as np
import pytest

import edmd_fixtures as F
from conftest import bits

pytestmark = pytest.mark.gpu

WALLS = dict(wall_x=1, wall_y=1, res_wall=0.9, add_field=1, field=-0.02)


@pytest.mark.parametrize("n, params, ncoll", [
    (40, {}, 300),        # long chains: a few disks meet again and again
    (400, {}, 0),
    (400, {}, 1),
    (400, {}, 63),
    (400, {}, 64),
    (400, {}, 65),
    (400, {}, 128),
    (400, {}, 1000),
    (400, WALLS, 500),
    (1200, {}, 3000),     # two disks share a slot of the table
    (1365, {}, 1500),     # the largest vector in LDS
    (1366, {}, 1500),     # the smallest in HBM
    (2500, WALLS, 3000),
])
@pytest.mark.parametrize("every", [0, 100])
def test_rounds_match_oracle(gpu, oracle, n, params, ncoll, every):
    if params:
        states = [F.walled_state(n, 0.5, 70 + k, wall_x=True, wall_y=True) for k in range(2)]
    else:
        states = [F.lattice_state(n, 0.6, seed=70 + k, lattice="fit") for k in range(2)]
    b = gpu.Batch(states, **params)
    b.deriv_begin(checkpoint_every=every, tape_capacity=0 if every else ncoll + 1)
    b.deriv_run(max_collisions=ncoll)
    rng = np.random.default_rng(n + ncoll)
    tin = [rng.standard_normal((n, 4)) for _ in states]
    lam = [rng.standard_normal((n, 4)) for _ in states]
    lw, lt = rng.uniform(0.5, 2.0, 2), rng.uniform(-3.0, 3.0, 2)
    tout, dw, dtl = b.tangent(tin)
    grad = b.adjoint(lw, lt, lam)
    for k, st in enumerate(states):
        o = oracle.Oracle(st, **params)
        s0 = o.state()
        o.tape_enable(ncoll + 16)
        o.run_collisions(ncoll)
        tape = o.tape()
        assert len(tape) == ncoll
        tan = tin[k].copy()
        rdw, rdtl = oracle.tangent(st["m"], s0["t"], tape, o.t, tan)
        np.testing.assert_array_equal(bits(tout[k]), bits(tan), err_msg="tangent %d" % k)
        assert bits(dw[k]) == bits(rdw) and bits(dtl[k]) == bits(rdtl)
        g = oracle.adjoint(st["m"], s0["t"], tape, o.t, lw[k], lt[k], lam[k])
        np.testing.assert_array_equal(bits(grad[k]), bits(g), err_msg="adjoint %d" % k)


def free_bytes(gpu):
    """Of the runtime that the library runs on: torch loads one of its own."""
    free, total = C.c_size_t(), C.c_size_t()
    assert gpu.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_checkpoint_memory_is_given_back(gpu):
    """A taping holds no checkpoint of the one before that it does not use: a
    whole tape after a checkpointed one of the same capacity none, a shorter
    one its own."""
    st = F.lattice_state(400, 0.6, seed=4, lattice="fit")
    b = gpu.Batch([st] * 256)
    ev = 0

    def tape(every, events):
        nonlocal ev
        b.deriv_begin(checkpoint_every=every, tape_capacity=64)
        ev += events
        b.deriv_run(max_events=ev)
        return free_bytes(gpu)

    tape(64, 64)
    start = free_bytes(gpu)
    long = tape(64, 64 * 40)
    kept = start - long
    assert kept > 39 * 256 * 400 * 128  # 40 snapshots of the systems' records
    assert tape(64, 64 * 40) >= long - (64 << 20)
    assert tape(64, 64 * 4) >= start - kept // 8
    tape(64, 64 * 40)
    b.deriv_begin(checkpoint_every=0, tape_capacity=64)
    assert free_bytes(gpu) >= start - (64 << 20)
    b.close()
