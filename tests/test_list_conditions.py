"""The dt conditions of the force pass over cached lists: every listed pair sets
one, as calcForce over the cached neighbours does (sph.h:545-560; the lists are
those of their first use, dataLL.impl.h:186-188), also when r or h has changed
since the lists were built."""
import numpy as np
import pytest

import oracle
import sphdem as sd

pytestmark = pytest.mark.gpu

VISC = {"morris+artificial": sd.F_VISC_MORRIS | sd.F_VISC_ARTIFICIAL, "morris": sd.F_VISC_MORRIS,
        "monaghan": sd.F_VISC_MONAGHAN, "cleary+artificial": sd.F_VISC_CLEARY | sd.F_VISC_ARTIFICIAL}
# FP64 as the other passes' conditions; the mixed form's h and signal speeds are
# FP32 values (6e-8) of a few operations
REL = {sd.FP64: 1e-15, sd.MIXED: 1e-5}


def fresh(case, precision, steps):
    rng = np.random.default_rng(5)
    case.h *= 1.0 - 0.2 * rng.random(case.n)
    sim, orc = sd.Sim(case, precision=precision), oracle.Oracle(case)
    for x in (sim, orc):
        if steps:
            x.run(steps)
        else:
            x.reset()
    # slow: the conditions of two pairs differ by their h first
    vh = rng.normal(size=(case.n, 3)) * 1e-4
    vh[case.iam == sd.SPH_BOUNDARY] = 0.0
    state = {k: orc.get(k) for k in ("r", "h", "dens", "pdr2")}
    for x in (sim, orc):
        x.pairs(sd.PAIRS_SPH)  # the lists, at this r and h
        x.set("vhat", vh)
        for k in ("r", "h", "dens"):
            x.set(k, state[k])
        g = x.globals()
        g.newDt = case.params.maxdt
        x.set_globals(g)
    return sim, orc, rng, state


def after_lists(flags, precision, change, steps):
    """(the library's dt, the oracle's)"""
    case = sd.dambreak_case(nf=9)
    case.params.flags = (case.params.flags & ~(sd.F_VISC_MORRIS | sd.F_VISC_ARTIFICIAL)) | flags
    sim, orc, rng, state = fresh(case, precision, steps)
    r, h = state["r"], state["h"]
    if "h" in change:
        h = h * (1.0 - 0.5 * rng.random(h.shape))
    if "r" in change:
        r = r + 0.8 * case.params.psep * (rng.random(r.shape) - 0.5)
    for x in (sim, orc):
        x.set("r", r)
        x.set("h", h)
        x.pass_("eos")
    orc.refresh_ghosts()
    p = np.asarray(orc.pairs(sd.PAIRS_SPH), np.int64)
    d2 = ((r[p[:, 0]] - r[p[:, 1]]) ** 2).sum(axis=1)
    outside = int((d2 > (2.0 * np.maximum(h[p[:, 0]], h[p[:, 1]])) ** 2).sum())
    assert outside > 0  # listed pairs beyond the radius of now
    for x in (sim, orc):
        x.pass_("force")
    return sim.reduce_dt(), orc.new_dt()


@pytest.mark.parametrize("precision", [sd.FP64, sd.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("change", ["h", "r", "rh"])
@pytest.mark.parametrize("visc", sorted(VISC))
def test_every_listed_pair_sets_a_condition(visc, change, precision):
    got, want = after_lists(VISC[visc], precision, change, 0)
    assert got == pytest.approx(want, rel=REL[precision])


@pytest.mark.parametrize("visc", sorted(VISC))
def test_the_lists_of_a_step_too(visc):
    """After a run the lists are those of its last reset, whatever search made
    them."""
    got, want = after_lists(VISC[visc], sd.FP64, "h", 1)
    assert got == pytest.approx(want, rel=1e-12)
