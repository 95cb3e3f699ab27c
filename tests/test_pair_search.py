"""The pair searches taken by groups of lanes (a sphere's or a fluid particle's
candidates side by side) and their device-side offsets: every kind's set equals
the oracle's over coupling radii of few and many sphere cells (the range of
cells a fluid particle's search keeps follows their ratio), with one query, with
numbers of queries around a workgroup's and a scan tile's, and with all spheres
in one corner (columns longer than a group) across the periodic faces; and the
triples of one query stay together, queries in the store's order."""
import numpy as np
import pytest

import oracle
import sphdem as sd

pytestmark = pytest.mark.gpu

KINDS = (sd.PAIRS_SPH, sd.PAIRS_DEM, sd.PAIRS_SPH2DEM, sd.PAIRS_DEM2SPH)


def same_sets(case):
    sim, orc = sd.Sim(case), oracle.Oracle(case)
    for kind in KINDS:
        g, o = np.asarray(sim.pairs(kind), np.int64), np.asarray(orc.pairs(kind), np.int64)
        assert len(g) == len(o), kind
        assert np.array_equal(np.unique(g, axis=0), np.unique(o, axis=0)), kind
        change = np.flatnonzero(np.diff(g[:, 0])) if len(g) else []
        assert len(np.unique(g[:, 0])) == (len(change) + 1 if len(g) else 0), kind
    sim.close()


@pytest.mark.parametrize("ratio", [2.5, 4.0, 9.0, 12.0, 16.0])
def test_coupling_radii_of_few_and_many_sphere_cells(ratio):
    """ratio: the coupling radius over the sphere search radius."""
    c = sd.sediment_case(nf=12, n_dem=90, seed=5)
    c.params.dem_search_radius = c.params.coupling_radius / ratio
    c.h[c.iam == sd.DEM] = c.params.dem_search_radius
    same_sets(c)


@pytest.mark.parametrize("n_dem", [1, 3, 15, 17, 64, 257])
def test_numbers_of_queries(n_dem):
    same_sets(sd.sediment_case(nf=12, n_dem=n_dem, seed=n_dem))


@pytest.mark.parametrize("nf", [10, 16, 19])  # below and above one and two scan tiles
def test_numbers_of_targets(nf):
    same_sets(sd.sediment_case(nf=nf, nz=12, n_dem=40, seed=nf))


def test_spheres_in_a_corner_across_the_periodic_faces():
    c = sd.sediment_case(nf=12, n_dem=200, seed=9)
    dem = np.flatnonzero(c.iam == sd.DEM)
    rng = np.random.default_rng(3)
    lo = np.array([c.params.rmin[d] for d in range(3)])
    L = np.array([c.params.rmax[d] for d in range(3)]) - lo
    p = rng.normal(scale=0.02, size=(len(dem), 3)) * L
    p[:, 2] = np.abs(p[:, 2]) + 0.3 * L[2]
    p[:, :2] = np.mod(p[:, :2], L[:2])
    c.r[dem] = lo + p
    same_sets(c)


@pytest.mark.parametrize("n_dem", [120, 128, 129, 300])
def test_queries_with_more_pairs_than_the_count_keeps(n_dem):
    """All spheres within a coupling radius of one fluid particle: queries with
    fewer pairs than the 128 the count keeps, that many, and more."""
    c = sd.sediment_case(nf=12, n_dem=n_dem, seed=4)
    dem = np.flatnonzero(c.iam == sd.DEM)
    rng = np.random.default_rng(n_dem)
    c.r[dem] = np.array([0.5, 0.5, 0.5]) + rng.normal(scale=0.01, size=(n_dem, 3))
    sim = sd.Sim(c)
    most = max(np.unique(np.asarray(sim.pairs(sd.PAIRS_SPH2DEM))[:, 0], return_counts=True)[1])
    assert most == n_dem
    sim.close()
    same_sets(c)
