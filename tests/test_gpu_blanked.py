"""Blanked particles in every path of the interaction: they stay where they were blanked, with whatever
position made them so, and no mechanical sum takes them."""
import numpy as np
import pytest

import pymfc
from parity import equal

pytestmark = pytest.mark.gpu

FIELDS = ["pos", "vel", "S", "rho", "T", "eps_pl", "fc", "ft", "flags", "id"]


def blanked_ids(s):
    return set(s.field("id")[(s.field("flags") & pymfc.FLAG_BLANKED) != 0].tolist())


@pytest.mark.parametrize("component", [0, 1])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_fp32c_blanked_particles_stay_excluded(component, value):
    """A rate of one workpiece particle that is not finite blanks it and the particles of the
    workpiece in whose support it lies in that step, and nothing after that, for every number of threads
    per particle (a particle moves by less than 1 % of its support radius in the steps in between)."""
    cfg = pymfc.cut_config(61, 17, 10.0, thermal="contact", speed_m_min=1000.0, jitter=0.01,
                           precision=pymfc.PREC_FP32C)
    runs = []
    for lanes, limit in ((1, 0), (4, 0), (8, 0), (1, 1)):
        g = pymfc.Sim(cfg)
        g.set_tuning(lanes=lanes, stage_limit=limit)
        g.step(10)
        ids, fl, pos, h, vt = (g.field(f) for f in ("id", "flags", "pos", "h", "vel_t"))
        free = np.sort(ids[fl == 0])
        hit = np.nonzero(ids == free[free.size // 2])[0][0]
        vt[hit, component] = value
        g.set_field("vel_t", vt)
        g.step(12)
        q = np.hypot(*(pos - pos[hit]).T) / (2 * h)
        wp = (fl & pymfc.FLAG_TOOL) == 0
        assert set(ids[wp & (q < 0.99)].tolist()) <= blanked_ids(g) <= set(ids[wp & (q < 1.01)].tolist()), lanes
        runs.append(g)
    for g in runs[1:]:
        for f in FIELDS:
            assert equal(runs[0].field(f), g.field(f)), f
