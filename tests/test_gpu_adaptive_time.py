"""The adaptive grid's own work at a size where one work-group can't do it."""
import pytest

import pymfc
from test_gpu_lanes import step_time

pytestmark = pytest.mark.gpu


def test_adaptive_grid_costs_a_part_of_the_step():
    """A step of 131k particles beside one on the locked grid: the box of the positions is found by one
    work-group (3 MB read, some 70 us), the binning by all: 1.8 times as long in all, 4 with the binning by
    that one work-group."""
    sims = [pymfc.Sim(pymfc.config_impact(200, adaptive=a)) for a in (True, False)]
    times = [step_time(s) for s in sims]
    assert times[0] < 2.2 * times[1], times
