"""The interaction over patches of cells: every number of threads per particle, and the path over the
records in memory that takes what a patch's LDS copy does not (too many candidates, columns too
dense for the masks, records that are not finite, an h that is not uniform, and entries past the
launch's work items), against the oracle bit for bit (FP64) or each other (FP32C)."""
import numpy as np
import pytest

import pymfc
import oracle_binding as ob
from parity import assert_bitwise, equal

pytestmark = pytest.mark.gpu

FIELDS = ["pos", "vel", "S", "rho", "p", "T", "eps_pl", "fc", "ft", "n", "R", "flags", "id", "hash"]


def cut(prec=pymfc.PREC_FP64, thermal="contact", nx=61, ny=17, **kw):
    return pymfc.cut_config(nx, ny, 10.0, thermal=thermal, speed_m_min=1000.0, jitter=0.01, precision=prec, **kw)


@pytest.mark.parametrize("lanes", [1, 4, 8])
@pytest.mark.parametrize("thermal", ["adiabatic", "contact", "pse"])
def test_lanes_match_the_oracle(lanes, thermal):
    cfg = cut(thermal=thermal)
    g, o = pymfc.Sim(cfg), ob.OracleSim(cfg)
    g.set_tuning(lanes=lanes)
    assert g.tuning()["lanes"] == lanes
    g.step(41)
    o.step(41)
    assert_bitwise(g, o, context=f"lanes {lanes}")
    assert equal(g.force_history(), o.force_history())


@pytest.mark.parametrize("thermal", ["adiabatic", "contact", "pse"])
def test_fp32c_bits_do_not_depend_on_lanes(thermal):
    cfg = cut(pymfc.PREC_FP32C, thermal=thermal)
    runs = []
    for lanes, limit in ((1, 0), (4, 0), (8, 0), (1, 1), (8, 1), (1, 400)):
        g = pymfc.Sim(cfg)
        g.set_tuning(lanes=lanes, stage_limit=limit)
        g.step(41)
        runs.append(g)
    for g in runs[1:]:
        for f in FIELDS:
            assert equal(runs[0].field(f), g.field(f)), f
        assert equal(runs[0].force_history(), g.force_history())


def test_lanes_change_between_steps():
    cfg = cut()
    g, o = pymfc.Sim(cfg), ob.OracleSim(cfg)
    for lanes in (1, 8, 4, 0):
        g.set_tuning(lanes=lanes)
        g.step(9)
        o.step(9)
    assert_bitwise(g, o, context="lanes changed")
    with pytest.raises(pymfc.MfcError):
        g.set_tuning(lanes=2)


@pytest.mark.parametrize("lanes", [1, 4, 8])
def test_uneven_h(lanes):
    cfg = cut()
    g, o = pymfc.Sim(cfg), ob.OracleSim(cfg)
    g.set_tuning(lanes=lanes)
    h = g.field("h")
    h = h * (1.0 - 0.05 * (np.arange(h.size) % 3))
    for s in (g, o):
        s.set_field("h", h)
        s.step(10)
    assert_bitwise(g, o, context="uneven h")


@pytest.mark.parametrize("lanes", [1, 4, 8])
@pytest.mark.parametrize("place", ["scattered", "heaped"])
def test_unusual_densities(lanes, place):
    """Particles scattered over the whole grid fill many more patches than the initial lattice
    (entries past the work items, windows of a few candidates); particles heaped into a few cells
    fill several parts of a patch and more candidates than the LDS copy and the masks take."""
    cfg = pymfc.config_rings(24)
    g, o = pymfc.Sim(cfg), ob.OracleSim(cfg)
    g.set_tuning(lanes=lanes)
    rng = np.random.default_rng(7)
    N = g.N
    if place == "scattered":
        pos = np.stack([rng.uniform(-0.19, 0.19, N), rng.uniform(-0.075, 0.075, N)], axis=1)
    else:
        pos = np.stack([rng.uniform(0.01, 0.022, N), rng.uniform(-0.01, 0.01, N)], axis=1)
    for s in (g, o):
        s.set_field("pos", pos)
        s.step(3)
    assert_bitwise(g, o, context=place)


@pytest.mark.parametrize("lanes", [1, 4, 8])
def test_nonfinite_and_blanked_neighbours(lanes):
    cfg = cut(thermal="contact")
    g, o = pymfc.Sim(cfg), ob.OracleSim(cfg)
    g.set_tuning(lanes=lanes)
    for s in (g, o):
        s.step(10)
    vt = o.field("vel_t")
    free = np.nonzero(o.field("flags") == 0)[0]
    vt[free[free.size // 2], 0] = np.nan
    vt[free[free.size // 3], 1] = np.inf
    for s in (g, o):
        s.set_field("vel_t", vt)
        s.step(20)
    assert (o.field("flags") & pymfc.FLAG_BLANKED).sum() >= 1
    assert_bitwise(g, o, context="non-finite")


@pytest.mark.parametrize("thermal", ["adiabatic", "contact", "pse"])
def test_gradient_of_both_pull_paths(thermal):
    """The reverse step's pull from the LDS copy (both terms of a pair in one evaluation) and from the
    records in memory, over segments of unequal length. Each contribution differs by some tens of
    rounding errors, there are about 50 per particle and step, and 30 steps follow each other:
    30 * 50 * 50 * 1.1e-16 = 8e-12 of the largest component, and two decades for the cancellation
    within the sums."""
    cfg = cut(thermal=thermal)
    cfg.promote_fp64, cfg.secant_tol = 1, 1e-14
    grads = []
    for limit in (0, 1):
        g = pymfc.Sim(cfg)
        g.set_tuning(stage_limit=limit)
        g.step(30)
        F = g.vjp_forward(30, 13, 10, 30)
        grads.append((F, g.vjp_backward([1.0, 0.5])))
    assert equal(grads[0][0], grads[1][0])
    a, b = grads[0][1], grads[1][1]
    assert np.all(np.isfinite(a)) and np.abs(a).max() > 0
    assert np.abs(a - b).max() <= 1e-9 * np.abs(a).max()


@pytest.mark.parametrize("lanes", [1, 8])
@pytest.mark.parametrize("n,C,tol", [(0.34, 0.014, 1e-14), (0.97, 0.97, 1e-6), (1.0, 0.014, 1e-6), (0.34, 1.0, 1e-6),
                                     (1.3, 2.0, 1e-14)])
def test_returns_match_the_oracle(lanes, n, C, tol):
    """The return's secant with exponents on both sides of the bound below which no value on its way
    needs a special case, to its end and folding, by a wave and by a whole work-group."""
    cfg = cut(thermal="adiabatic")
    cfg.jc_n, cfg.jc_C, cfg.secant_tol = n, C, tol
    g, o = pymfc.Sim(cfg), ob.OracleSim(cfg)
    g.set_tuning(lanes=lanes)
    g.step(120)
    o.step(120)
    assert np.count_nonzero(o.field("eps_pl")) > 10
    assert_bitwise(g, o, context=f"n {n} C {C}")


@pytest.mark.parametrize("lanes,limit", [(0, 0), (1, 0), (0, 1)])
def test_gradient_with_recorded_returns(lanes, limit):
    """A replay that takes the secant results of the recorded run, and one that iterates again (a run
    so long that its tape would be larger than its checkpoints and slots; the steps past the window
    carry no adjoint): the same expressions on the same values, so the same bits. Steps after a
    recorded run write nothing to its tape."""
    cfg = cut(thermal="adiabatic")
    cfg.promote_fp64, cfg.secant_tol = 1, 1e-14
    grads = []
    for n, K in ((60, 13), (14000, 75)):
        g = pymfc.Sim(cfg)
        g.set_tuning(lanes=lanes, stage_limit=limit)
        g.step(60)
        F = g.vjp_forward(n, K, 10, 60)
        grads.append((F, g.vjp_backward([1.0, 0.5])))
        if n == 60:
            o = ob.OracleSim(cfg)
            o.step(140)
            g.step(20)
            assert np.count_nonzero(o.field("eps_pl")) > 10
            assert_bitwise(g, o, context="after a recorded run")
            assert equal(grads[0][1], g.vjp_backward([1.0, 0.5]))  # its tape is as it was
    assert equal(grads[0][0], grads[1][0])
    assert np.all(np.isfinite(grads[0][1])) and np.abs(grads[0][1]).max() > 0
    assert equal(grads[0][1], grads[1][1])
