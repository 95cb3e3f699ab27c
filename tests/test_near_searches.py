"""The step's list search where h really differs from particle to particle
(CONST_H: a step leaves h alone), where its room overflows and where it cannot
serve: results are those of the segmented search bit for bit, the near search is
the one that ran, and it is left off after it failed."""
import numpy as np
import pytest

import sphdem as sd

pytestmark = pytest.mark.gpu

FIELDS = ("r", "v", "vhat", "f", "dens", "h", "press", "porosity", "fdrag", "shepSum", "omega")


def periodic(nf):  # ghosts on two axes
    return lambda: sd.sediment_case(nf=nf, nz=max(nf, 12), n_dem=40, seed=nf)


def closed(nf):  # no ghosts
    return lambda: sd.dambreak_case(nf=nf, dx=0.32 / nf, seed=nf, with_dem=40, liq_dem_flags=True)


# nine wavefronts a tile up to 32768 targets, three beyond
SIZES = {"periodic13": periodic(13), "closed17": closed(17), "periodic34": periodic(34),
         "closed36": closed(36)}


def sph_group(case):
    return np.isin(case.iam, (sd.SPH, sd.SPH_BOUNDARY))


def spread(case, rng):
    """h over 0.7 to 1 of its value."""
    s = sph_group(case)
    case.h[s] *= 1.0 - 0.3 * rng.random(int(s.sum()))


def crowded(case, rng):
    """2.4 times the usual particles in the space, the cells larger by one corner
    particle's h (175 a cell, and psep unknown), the radius of all others small: the
    mask words overflow."""
    s = sph_group(case)
    c = case.r[s].mean(axis=0)
    case.r[s] = c + 0.75 * (case.r[s] - c)
    corner = np.flatnonzero(s)[np.argmin(case.r[s].sum(axis=1))]
    big = 1.4 * case.h[corner]
    case.params.psep = 0.0
    case.h[s] *= 0.85
    case.h[corner] = big


def long_lists(case, rng):
    """Twice the usual particles and a spread of h: near lists of over 256 entries
    where the pairs are fewer."""
    s = sph_group(case)
    c = case.r[s].mean(axis=0)
    case.r[s] = c + 0.8 * (case.r[s] - c)
    case.h[s] *= 1.0 - 0.12 * rng.random(int(s.sum()))


def run(sim, steps):
    sim.run(steps)


def run_graph(sim, steps):
    sim.run_graph(steps)


def run_many(sim, steps):
    other = sd.Sim(sd.sediment_case(nf=12, n_dem=20))
    sd.run_many([sim, other], steps)
    other.close()


def run_many_graph(sim, steps):
    other = sd.Sim(sd.sediment_case(nf=12, n_dem=20))
    sd.run_many([sim, other], steps, graph=True)
    other.close()


def states(make, edit, precision, how=run, steps=2, flags=None, drop=0):
    """Fields, globals, pairs, output variables of both searches, and what the near
    search did."""
    out, near = [], None
    for seg in (64, 0):
        case = make()
        case.params.flags = (case.params.flags & ~drop) | sd.F_CONST_H | (flags or 0)
        edit(case, np.random.default_rng(17))
        sim = sd.Sim(case, precision=precision)
        sim.set_tile_shape(seg, 256)
        (run if seg else how)(sim, steps)
        s = sph_group(case)
        assert np.array_equal(sim.get("h")[s & (sim.get("iam") != sd.DELETED)],
                              case.h[s & (sim.get("iam") != sd.DELETED)])
        near = sim.near_searches()
        assert near[0] == 0 or seg == 0
        g = sim.globals()
        vars_ = sim.output_vars()
        out.append(({k: sim.get(k) for k in FIELDS}, (g.dt, g.time, g.sphStep),
                    sim.pairs(sd.PAIRS_SPH), vars_))
        sim.close()
    return out, near


def check(out):
    (fa, ga, pa, va), (fb, gb, pb, vb) = out
    for k in FIELDS:
        assert np.array_equal(fa[k], fb[k], equal_nan=True), k
    assert ga == gb
    assert np.array_equal(pa, pb)
    for k in va:
        assert np.array_equal(np.asarray(va[k]), np.asarray(vb[k]), equal_nan=True), k


PRECISIONS = pytest.mark.parametrize("precision", [sd.FP64, sd.MIXED], ids=["fp64", "mixed"])


@PRECISIONS
@pytest.mark.parametrize("size", sorted(SIZES))
def test_h_that_differs(size, precision):
    out, (searches, exact) = states(SIZES[size], spread, precision)
    check(out)
    assert searches == 4 and exact == 0
    h = out[1][0]["h"]
    assert h.max() > 1.3 * h[h > 0.5 * h.max()].min()


@PRECISIONS
@pytest.mark.parametrize("edit", [crowded, long_lists])
@pytest.mark.parametrize("size", sorted(SIZES))
def test_targets_left_to_the_exact_search(size, edit, precision):
    out, (searches, exact) = states(SIZES[size], edit, precision, steps=1)
    check(out)
    assert searches > 0 and exact > 0


@PRECISIONS
@pytest.mark.parametrize("visc", [sd.F_VISC_MORRIS | sd.F_VISC_ARTIFICIAL,
                                  sd.F_VISC_CLEARY | sd.F_VISC_ARTIFICIAL, sd.F_VISC_MONAGHAN])
def test_conditions_of_each_pair_with_h_that_differs(visc, precision):
    """The signal speeds of pairs, entries that may be none among them."""
    def slow(case, rng):
        spread(case, rng)
        case.vhat[:] = 1e-4 * rng.normal(size=case.vhat.shape)
        case.vhat[case.iam == sd.SPH_BOUNDARY] = 0.0
        case.v[:] = case.vhat

    drop = sd.F_VISC_MORRIS | sd.F_VISC_ARTIFICIAL
    out, (searches, _) = states(lambda: sd.dambreak_case(nf=17), slow, precision, flags=visc,
                                drop=drop, steps=3)
    check(out)
    assert searches == 6


@pytest.mark.parametrize("how", [run_graph, run_many, run_many_graph])
@PRECISIONS
@pytest.mark.parametrize("size", ["periodic13", "closed17", "periodic34"])
def test_replayed_and_ensemble_steps(size, precision, how):
    out, (searches, exact) = states(SIZES[size], spread, precision, how=how, steps=5)
    check(out)
    assert searches >= 10 and exact == 0  # a capture may follow a step run as launches


@PRECISIONS
@pytest.mark.parametrize("nf", [12, 28])
def test_an_h_of_zero(nf, precision):
    """No record is a bound: every target is left to the exact part, and, beyond 32768
    of them, the next resets search exactly from the start."""
    def zero(case, rng):
        s = sph_group(case)
        i = np.flatnonzero(case.iam == sd.SPH)[0]
        top = case.r[s].max(axis=0)
        case.r[i] = [0.75 * top[0], 0.5 * top[1], 0.5 * top[2]]
        case.h[i] = 0.0

    out, (searches, exact) = states(lambda: sd.dambreak_case(nf=nf), zero, precision, steps=3)
    check(out)
    n = int(sph_group(sd.dambreak_case(nf=nf)).sum())
    assert searches == (6 if n <= 32768 else 1)
    assert exact == searches * n


def test_the_near_search_waits_after_it_failed():
    """Crowded cells that the initial spacing does not tell of, beyond 32768 targets:
    one attempt, sixteen resets of exact searches, another, thirty-two."""
    case = sd.dambreak_case(nf=28)
    case.params.flags |= sd.F_CONST_H
    case.params.psep = 0.0
    case.h[np.flatnonzero(case.iam == sd.SPH_BOUNDARY)[0]] *= 2.0
    sim = sd.Sim(case)
    seen = []
    for _ in range(30):
        sim.run(1)
        seen.append(sim.near_searches()[0])
    assert seen[0] == 1 and seen[7] == 1 and seen[8] == 2 and seen[-1] == 3
    sim.close()
