"""Arrays to and from the card in pieces: states at the edges of a piece
(half a megabyte of 64-byte records), batches whose arrays are sent in several
pieces, and a taping that takes over the memory of the one before."""
import numpy as np
import pytest

import edmd_fixtures as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 8191, 8192, 8193, 24577])
def test_state_and_events_in_pieces(gpu, oracle, n):
    st = F.lattice_state(n, 0.02 if n < 10 else 0.6, seed=n, lattice="fit")
    h = gpu.System(st)
    o = oracle.Oracle(st)
    s, so = h.state(), o.state()
    n = len(st["x"])
    for k in ("x", "y", "vx", "vy"):
        assert len(s[k]) == n and np.array_equal(s[k], so[k]), k
    assert np.array_equal(h.radii(), st["rad"])
    b = gpu.Batch([st, st])
    for k in range(2):
        assert np.array_equal(b.state(k)["vx"], st["vx"])
        e, e0 = b.events(k), h.events()
        for f in ("t_coll", "partner", "t_cross", "dir"):
            assert np.array_equal(e[f], e0[f]), f


def test_batch_sent_in_several_pieces(gpu):
    """Five systems of 70000 disks (22 MB of records) and small ones between."""
    big, small = F.lattice_state(70000, 0.5, seed=1), F.lattice_state(300, 0.5, seed=2)
    states = [big, small, big, big, small, big, big, small]
    b = gpu.Batch(states)
    alone = {300: gpu.System(small).events(), 70000: gpu.System(big).events()}
    for k, st in enumerate(states):
        s = b.state(k)
        for f in ("vx", "vy"):
            assert np.array_equal(s[f], st[f]), (k, f)
        e, e0 = b.events(k), alone[70000 if st is big else 300]
        assert np.array_equal(e["t_coll"], e0["t_coll"]) and np.array_equal(e["partner"], e0["partner"])


@pytest.mark.parametrize("first,second", [((0, 600), (0, 600)), ((64, 0), (64, 0)), ((0, 300), (300, 0)),
                                          ((64, 0), (0, 700))])
def test_taping_again(gpu, first, second):
    """(checkpoint_every, tape_capacity) of two tapings of one batch: the
    second one's gradient is that of a batch that was taped once."""
    states = [F.lattice_state(200, 0.55, seed=k, lattice="fit") for k in range(3)]
    out = []
    for tapings in ((first, second), (second,)):
        b = gpu.Batch(states)
        done = 300 * (3 - len(tapings))
        b.run(max_collisions=done)
        for every, cap in tapings:
            b.deriv_begin(checkpoint_every=every, tape_capacity=cap)
            done += 300
            b.deriv_run(max_collisions=done)
        out.append(np.concatenate(b.adjoint(lw=1.0)))
    assert np.array_equal(out[0], out[1])
