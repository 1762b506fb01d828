"""Particles spread over many more patches of cells than the body they came from."""
import numpy as np
import pytest

import pymfc
import oracle_binding as ob
from parity import assert_bitwise, equal
from test_gpu_lanes import step_time

pytestmark = pytest.mark.gpu


def scenario(name, prec=pymfc.PREC_FP64):
    if name.startswith("rings"):
        cfg = pymfc.config_rings(60, prec)
    else:
        cfg = pymfc.cut_config(90, 30, 10.0, thermal=name[4:], jitter=0.01, precision=prec)
    if name == "rings_rothlin":
        cfg.grid_kind = pymfc.GRID_ROTHLIN
    return cfg


def scatter(s, share, seed=3):
    """a share of the free particles anywhere in the grid"""
    rng = np.random.default_rng(seed)
    i, pos = s.info, s.field("pos")
    hit = (s.field("flags") == 0) & (rng.uniform(size=s.N) < share)
    box = np.array([i.grid_nx, i.grid_ny]) * i.cell_size
    at = np.array([i.bbmin_x, i.bbmin_y]) + box * rng.uniform(0.02, 0.98, (s.N, 2))
    s.set_field("pos", np.where(hit[:, None], at, pos))


@pytest.mark.parametrize("lanes", [1, 4, 8])
@pytest.mark.parametrize("name", ["rings", "rings_rothlin", "cut_contact", "cut_pse"])
@pytest.mark.parametrize("share", [0.02, 0.1, 1.0])
def test_scattered_particles(lanes, name, share):
    """Entries past the work items and, past 1.3 times as many, tiles of the sorted order."""
    cfg = scenario(name)
    g, o = pymfc.Sim(cfg), ob.OracleSim(cfg)
    g.set_tuning(lanes=lanes)
    for s in (g, o):
        scatter(s, share)
        s.step(3)
    assert_bitwise(g, o, context=f"{share} of {name}")
    assert equal(g.cells(), o.cells())


@pytest.mark.parametrize("name", ["rings", "cut_pse"])
def test_scattered_fp32c_bits_do_not_depend_on_lanes(name):
    runs = []
    for lanes in (1, 4, 8):
        g = pymfc.Sim(scenario(name, pymfc.PREC_FP32C))
        g.set_tuning(lanes=lanes)
        scatter(g, 0.3)
        g.step(3)
        runs.append(g)
    for g in runs[1:]:
        for f in ("pos", "vel", "S", "rho", "T", "flags", "id"):
            assert equal(runs[0].field(f), g.field(f)), f


@pytest.mark.parametrize("lanes", [1, 4])
def test_scattered_particles_take_no_longer(lanes):
    """Particles with hardly a neighbour, in ten times as many patches: with a work-group for each patch, one
    behind the other, their step took six times as long as the body's, by tiles about as long."""
    sims = [pymfc.Sim(pymfc.config_rings(200)) for _ in range(2)]
    scatter(sims[1], 1.0)
    for s in sims:
        s.set_tuning(lanes=lanes)
        s.set_field("vel", np.zeros((s.N, 2)))
    times = [step_time(s, 32) for s in sims]
    assert times[1] < 2.0 * times[0], times
