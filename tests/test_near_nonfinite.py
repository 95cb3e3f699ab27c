"""A particle whose density or mass is infinite or NaN (and whose h stays as it
is, CONST_H) reaches the sums of its neighbours only, whichever search made the
lists: a step's results are the same bit for bit, deletions included."""
import numpy as np
import pytest

import sphdem as sd

pytestmark = pytest.mark.gpu

FIELDS = ("r", "v", "vhat", "f", "fp", "fv", "dens", "dddt", "h", "press", "omega", "iam")


def dam():  # artificial viscosity, plain omega
    return sd.dambreak_case(nf=13)


def coupled():  # omega fused into the walks
    return sd.dambreak_case(nf=13, dx=0.32 / 13, with_dem=30, liq_dem_flags=True)


def monaghan():
    c = sd.dambreak_case(nf=13)
    c.params.flags = (c.params.flags & ~(sd.F_VISC_MORRIS | sd.F_VISC_ARTIFICIAL)) \
        | sd.F_VISC_MONAGHAN
    return c


def periodic():
    return sd.sediment_case(nf=13, n_dem=30, seed=2)


def step(make, field, value, precision, seg, how="run", steps=1):
    case = make()
    case.params.flags |= sd.F_CONST_H
    rng = np.random.default_rng(8)
    sph = np.isin(case.iam, (sd.SPH, sd.SPH_BOUNDARY))
    # uneven h: lists then hold entries well outside the radius
    case.h[sph] *= 1.0 - 0.3 * rng.random(int(sph.sum()))
    case.vhat[case.iam == sd.SPH] = 0.05 * rng.normal(size=(int((case.iam == sd.SPH).sum()), 3))
    case.v[:] = case.vhat
    sim = sd.Sim(case, precision=precision)
    sim.set_tile_shape(seg, 256)
    a = sim.get(field)
    mid = case.r[case.iam == sd.SPH].mean(axis=0)
    hit = [int(np.argmin(((case.r - mid) ** 2).sum(axis=1) + 1e9 * ~sph)),
           int(np.flatnonzero(case.iam == sd.SPH_BOUNDARY)[11])]
    a[hit] = value
    sim.set(field, a)
    getattr(sim, how)(steps)
    out = {k: sim.get(k) for k in FIELDS}
    out["deleted"] = sim.num_deleted()
    out["dt"] = sim.globals().dt
    sim.close()
    return out


@pytest.mark.parametrize("precision", [sd.FP64, sd.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("field, value", [("dens", np.nan), ("dens", np.inf), ("dens", 0.0),
                                          ("mass", np.inf), ("mass", np.nan)])
@pytest.mark.parametrize("make", [dam, coupled, monaghan, periodic])
def test_a_value_that_is_not_finite_stays_within_its_radius(make, field, value, precision):
    exact, near = (step(make, field, value, precision, seg) for seg in (64, 0))
    for k in exact:
        assert np.array_equal(exact[k], near[k], equal_nan=True), k
    assert not np.all(np.isfinite(near["f"])) or near["deleted"] or value == 0.0


@pytest.mark.parametrize("precision", [sd.FP64, sd.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("make", [coupled, periodic])
def test_replayed_steps_too(make, precision):
    """The flag words of a step's two searches change places from search to search: in
    a replayed step as in the one captured."""
    exact = step(make, "mass", np.inf, precision, 64, steps=4)
    near = step(make, "mass", np.inf, precision, 0, how="run_graph", steps=4)
    for k in exact:
        assert np.array_equal(exact[k], near[k], equal_nan=True), k
