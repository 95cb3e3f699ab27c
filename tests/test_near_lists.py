"""The step's own list search (near lists: every pair and a few entries beyond
its radius, whose terms are zero) against the segmented search (the FP64 test
on every candidate): a step's results are the same bit for bit, and so are the
pair lists asked for after it."""
import numpy as np
import pytest

import sphdem as sd

pytestmark = pytest.mark.gpu

FIELDS = ("r", "v", "vhat", "f", "dens", "h", "press", "porosity", "fdrag", "shepSum", "omega")


def periodic(nf):  # ghosts on two axes
    return lambda: sd.sediment_case(nf=nf, nz=max(nf, 12), n_dem=40, seed=nf)


def closed(nf):  # no ghosts
    return lambda: sd.dambreak_case(nf=nf, dx=0.32 / nf, seed=nf, with_dem=40, liq_dem_flags=True)


def viscosity(mk, flag):
    def make():
        c = mk()
        c.params.flags = (c.params.flags & ~sd.F_VISC_MORRIS) | flag
        return c
    return make


def spread(by):
    """h over [1 - by, 1] of its value: the larger h of the two decides a pair."""
    def edit(sim, draws):
        h = sim.get("h")
        sim.set("h", h * (1.0 - by * draws(h.shape)))
    return edit


def dense(by):
    """Twice the usual particles a cell, and a larger cell (one corner particle's
    h): word and list overflow."""
    def edit(sim, draws):
        r, h = sim.get("r"), sim.get("h")
        sph = np.isin(sim.get("iam"), (sd.SPH, sd.SPH_BOUNDARY))
        c = r[sph].mean(axis=0)
        r[sph] = c + 0.8 * (r[sph] - c)
        h = h * (1.0 - by * draws(h.shape))
        corner = np.flatnonzero(sph)[np.argmin(r[sph].sum(axis=1))]
        h[corner] *= 1.15
        sim.set("r", r)
        sim.set("h", h)
    return edit


def zero_h(sim, draws):
    """A particle alone in the open part of the box with h = 0: no record is a bound."""
    r, h = sim.get("r"), sim.get("h")
    i = np.flatnonzero(sim.get("iam") == sd.SPH)[0]
    sph = np.isin(sim.get("iam"), (sd.SPH, sd.SPH_BOUNDARY))
    top = r[sph].max(axis=0)
    r[i] = [0.75 * top[0], 0.5 * top[1], 0.5 * top[2]]
    h[i] = 0.0
    sim.set("r", r)
    sim.set("h", h)


# targets from one tile to past the nine-wavefront form's range
SIZES = {"periodic8": periodic(8), "periodic13": periodic(13), "periodic34": periodic(34),
         "closed9": closed(9), "closed17": closed(17), "closed36": closed(36)}


def states(mk, edit, precision, steps=2):
    out = []
    for seg in (64, 0):
        d = np.random.default_rng(17)
        sim = sd.Sim(mk(), precision=precision)
        sim.set_tile_shape(seg, 256)
        if edit:
            edit(sim, d.random)
        sim.run(steps)
        g = sim.globals()
        out.append(({nm: sim.get(nm) for nm in FIELDS}, (g.dt, g.time),
                    sim.pairs(sd.PAIRS_SPH)))
        sim.close()
    return out


def check(mk, edit, precision):
    (fa, ga, pa), (fb, gb, pb) = states(mk, edit, precision)
    for nm in FIELDS:
        assert np.array_equal(fa[nm], fb[nm], equal_nan=True), nm
    assert ga == gb
    assert np.array_equal(pa, pb)


@pytest.mark.parametrize("precision", [sd.FP64, sd.MIXED])
@pytest.mark.parametrize("size", sorted(SIZES))
def test_a_step_does_not_depend_on_the_search(size, precision):
    check(SIZES[size], None, precision)


@pytest.mark.parametrize("precision", [sd.FP64, sd.MIXED])
@pytest.mark.parametrize("edit", [spread(0.02), spread(0.3), dense(0.0), dense(0.1)],
                         ids=["h2", "h30", "dense", "dense_h10"])
@pytest.mark.parametrize("size", ["periodic13", "closed17", "closed36"])
def test_uneven_h_and_crowded_cells(size, edit, precision):
    check(SIZES[size], edit, precision)


@pytest.mark.parametrize("precision", [sd.FP64, sd.MIXED])
def test_an_h_of_zero_leaves_every_target_to_the_exact_search(precision):
    check(lambda: sd.dambreak_case(nf=12), zero_h, precision)


@pytest.mark.parametrize("precision", [sd.FP64, sd.MIXED])
@pytest.mark.parametrize("flag", [sd.F_VISC_MONAGHAN, sd.F_VISC_CLEARY])
def test_the_dt_conditions_take_pairs_only(flag, precision):
    check(viscosity(SIZES["closed17"], flag), spread(0.3), precision)


@pytest.mark.parametrize("change", ["r", "h", "both", "start", "h then start"])
@pytest.mark.parametrize("size", ["periodic13", "closed17"])
def test_pairs_after_a_step_are_those_of_its_lists(size, change):
    """r or h set, or a half-step started, after a run: the pairs stay those of the
    last reset's lists, whichever search made them."""
    got = []
    for seg in (64, 0):
        sim = sd.Sim(SIZES[size]())
        sim.set_tile_shape(seg, 256)
        spread(0.2)(sim, np.random.default_rng(3).random)
        sim.run(2)
        d = np.random.default_rng(4)
        if change in ("r", "both"):
            r = sim.get("r")
            sim.set("r", r + 1e-3 * (d.random(r.shape) - 0.5))
        if change in ("h", "both", "h then start"):
            h = sim.get("h")
            sim.set("h", h * (0.8 + 0.1 * d.random(h.shape)))
        if "start" in change:
            sim.start()
        p = sim.pairs(sd.PAIRS_SPH)
        sim.run(1)
        got.append((p, sim.get("dens"), sim.get("r"), sim.pairs(sd.PAIRS_SPH)))
        sim.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
