"""The event loops against one another where they part: the state that a full
cell leaves behind (addToCell, EDMD.c:2576-2585, has no bound; the capacity is
this library's)."""
import numpy as np
import pytest

import edmd_fixtures as F
from test_gpu_wide import QUIET, same_state, same_trace

pytestmark = pytest.mark.gpu


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
