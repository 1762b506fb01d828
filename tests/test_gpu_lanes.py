"""The number of threads per particle is a launch setting: changing it changes no result."""
import time

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


def cut(prec=pymfc.PREC_FP64, hdx=1.5, nx=61, ny=17, thermal="contact", **kw):
    cfg = pymfc.cut_config(nx, ny, 10.0, thermal=thermal, speed_m_min=1000.0, jitter=0.01, precision=prec, **kw)
    cfg.hdx = hdx
    return cfg


def uneven(s):
    h = s.field("h")
    s.set_field("h", h * (1.0 - 0.05 * (s.field("id") % 3)))


@pytest.mark.parametrize("thermal", ["contact", "pse"])
@pytest.mark.parametrize("hdx", [1.0, 2.1, 2.8, 3.4, 6.0])
@pytest.mark.parametrize("lanes", [1, 4, 8])
def test_smoothing_lengths(lanes, hdx, thermal):
    """From less than one to many lattice points per cell: windows whose columns hold up to 32, 64 and 160
    candidates and more, and windows of more candidates than a patch's copy of whole records, or of
    their parts, has room for; also with an h of its own for each particle."""
    g, o = pymfc.Sim(cut(hdx=hdx, thermal=thermal)), ob.OracleSim(cut(hdx=hdx, thermal=thermal))
    g.set_tuning(lanes=lanes)
    for s in (g, o):
        s.step(9)
    assert_bitwise(g, o, context=f"hdx {hdx}")
    for s in (g, o):
        uneven(s)
        s.step(9)
    assert_bitwise(g, o, context=f"hdx {hdx}, uneven h")


@pytest.mark.parametrize("hdx", [1.5, 2.3])
def test_fp32c_bits_do_not_depend_on_lanes_or_stage(hdx):
    runs = []
    for lanes, limit in ((1, 0), (4, 0), (8, 0), (1, 1)):
        g = pymfc.Sim(cut(pymfc.PREC_FP32C, hdx=hdx))
        g.set_tuning(lanes=lanes, stage_limit=limit)
        g.step(9)
        uneven(g)
        g.step(9)
        runs.append(g)
    for g in runs[1:]:
        for f in ("pos", "vel", "S", "rho", "T", "fc", "ft", "id"):
            assert equal(runs[0].field(f), g.field(f)), f


@pytest.mark.parametrize("batch", [False, True])
def test_kernel_follows_the_h_of_the_state(batch):
    """h written between blocks of steps that replay captured graphs, to one of its own for each
    particle and back, in a handle or in one instance of a batch."""
    cfgs = [cut(), cut(hdx=2.3), cut(nx=41)] if batch else [cut()]
    handle = pymfc.Batch(cfgs) if batch else pymfc.Sim(cfgs[0])
    sims = list(handle.instances) if batch else [handle]
    oracles = [ob.OracleSim(c) for c in cfgs]
    h0 = sims[0].field("h")
    for block in range(3):
        for s in (handle, *oracles):
            s.step(19)
        for s, o in zip(sims, oracles):
            assert_bitwise(s, o, context=f"block {block}")
        for s in (sims[0], oracles[0]):
            if block == 0:
                uneven(s)
            else:
                s.set_field("h", h0)


def step_time(s, n=64):
    s.step(32)
    best = np.inf
    for _ in range(5):
        s.sync()
        t = time.perf_counter()
        s.step(n)
        s.sync()
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("prec", [pymfc.PREC_FP64, pymfc.PREC_FP32C])
def test_uneven_h_costs_little_time(prec):
    """The same pairs and some loads more: 1.6 times as long at most (by themselves from the records in
    memory, the pairs take 2.2 to 2.8 times as long)."""
    sims = [pymfc.Sim(pymfc.cut_config(750, 200, 2.0, thermal="contact", jitter=0.01, precision=prec)) for _ in range(2)]
    uneven(sims[1])
    times = [step_time(s) for s in sims]
    assert times[1] < 1.6 * times[0], times


@pytest.mark.parametrize("lanes", [1, 4, 8])
@pytest.mark.parametrize("name", ["rothlin", "impact", "rings", "tanh_jc"])
def test_scenarios(lanes, name):
    """The cell ranges of the rothlin grid, whose sort leaves the friction force in place, an adaptive
    grid, a body without a tool and the tanh flow stress, whose secant takes other lanes."""
    if name == "impact":
        cfg = pymfc.config_impact(20)
    elif name == "rings":
        cfg = pymfc.config_rings(24)
    else:
        cfg = cut(nx=40, ny=12)
        if name == "rothlin":
            cfg.grid_kind = pymfc.GRID_ROTHLIN
        else:
            cfg.jc_model = pymfc.JC_TANH
            cfg.jc_tanh_a, cfg.jc_tanh_b, cfg.jc_tanh_c, cfg.jc_tanh_d = 2.0, 5.0, 1.0, 0.5
    g, o = pymfc.Sim(cfg), ob.OracleSim(cfg)
    g.set_tuning(lanes=lanes)
    for _ in range(3):
        g.step(33)
        o.step(33)
        assert_bitwise(g, o, context=name)
    assert equal(g.force_history(), o.force_history())
    assert equal(g.cells(), o.cells())


@pytest.mark.parametrize("prec", [pymfc.PREC_FP64, pymfc.PREC_FP32C])
@pytest.mark.parametrize("lanes", [1, 4, 8])
def test_mixed_batches(lanes, prec):
    """Cuts of every thermal model beside the bodies, an adaptive grid, the rothlin grid and dense cells."""
    cfgs = [cut(prec, thermal="adiabatic"), cut(prec, nx=41), cut(prec, thermal="pse", nx=33), cut(prec, hdx=2.3, nx=33),
            pymfc.config_rings(24, prec), pymfc.config_impact(16, prec), cut(prec, nx=31)]
    cfgs[-1].grid_kind = pymfc.GRID_ROTHLIN
    b = pymfc.Batch(cfgs)
    b.set_tuning(lanes=lanes)
    b.step(21)
    for i, c in enumerate(cfgs):
        s = pymfc.Sim(c)
        s.step(21)
        for f in ("pos", "vel", "S", "T", "eps_pl", "fc", "ft", "flags", "id"):
            assert equal(b[i].field(f), s.field(f)), (i, f)
        assert equal(b[i].force_history(), s.force_history()), i


def test_autotuner_tries_kernels():
    """No two candidates of the default space are the same launches twice, but for lanes 0, which stands for
    one of the others; the threads per particle are among them."""
    s = pymfc.Sim(cut(nx=40, ny=12))
    t = pymfc.autotune(s, steps=2, rounds=1)
    assert {"lanes", "xcd_chunk"} == {k for k, v in pymfc.TUNING_SPACE.items() if len(v) > 1}
    assert set(pymfc.TUNING_SPACE["lanes"]) == {0, 1, 4, 8}
    assert s.tuning()["lanes"] == t["lanes"] and s.tuning()["xcd_chunk"] == t["xcd_chunk"]
