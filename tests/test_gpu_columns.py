"""States, radii and events read as arrays laid out by the card (from 4096
rows on) and as rows, at the edges of both and of the pieces (10064 rows of a
state's 52 bytes, 18704 of an event's 28, 65472 radii)."""
import numpy as np
import pytest

import edmd_fixtures as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4095, 4096, 4097, 10063, 10064, 10065, 18704, 18705, 65473])
def test_arrays_of_members(gpu, n):
    st = F.lattice_state(n, 0.5, seed=n, lattice="fit")
    rng = np.random.default_rng(n)
    st["rad"] = 0.5 - 0.01 * rng.random(n)
    h = gpu.System(st)
    s = h.state()
    for k in ("x", "y", "vx", "vy"):
        assert np.array_equal(s[k], st[k]), k
    assert np.array_equal(h.radii(), st["rad"])
    assert not s["t"].any() and not s["coll"].any()
    ncx, ncy, _, csx, csy = h.grid()
    assert np.array_equal(s["cx"], np.minimum((st["x"] * (1 / csx)).astype(np.int32), ncx - 1))
    assert np.array_equal(s["cy"], np.minimum((st["y"] * (1 / csy)).astype(np.int32), ncy - 1))
    # each leaf of the calendar is the earlier of its disk's two events
    e = h.events()
    b = gpu.Batch([st])
    leaf, code = (b.calendar(0)[k][:n] for k in ("key", "aux"))
    assert np.array_equal(leaf, np.minimum(e["t_coll"], e["t_cross"]))
    first = e["t_coll"] < e["t_cross"]
    assert np.array_equal(code[first], e["partner"][first])
    assert np.array_equal(code[e["t_cross"] < e["t_coll"]], -e["dir"][e["t_cross"] < e["t_coll"]])
    assert not e["coll_actual"].any()
