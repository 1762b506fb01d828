"""The number of threads per particle is a launch setting: changing it changes no result."""
import numpy as np
import pytest

import pymfc
import oracle_binding as ob
from parity import assert_bitwise, equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [False, True])
def test_out_of_grid_count_does_not_depend_on_lanes(batch):
    """A particle outside the grid is counted once per binned state, also where the threads per particle
    (and with them the shape of the patches) change in between: the count of a run left alone."""
    cfg = pymfc.cut_config(61, 17, 10.0, thermal="contact")
    o, alone = ob.OracleSim(cfg), pymfc.Sim(cfg)
    handle = pymfc.Batch([cfg, cfg]) if batch else pymfc.Sim(cfg)
    sims = handle.instances if batch else [handle]
    pos = o.field("pos")
    pos[0, 1] += 100.0
    for s in [o, alone] + list(sims):
        s.set_field("pos", pos)
    for s in (o, alone, handle):
        s.step(2)
    for lanes in (1, 4, 8, 4, 1):
        handle.set_tuning(lanes=lanes)
        for s in (o, alone, handle):
            s.step(3)
        for s in sims:
            assert s.info.out_of_grid == alone.info.out_of_grid > 0
            assert_bitwise(s, o, context=f"lanes {lanes}")
