"""The coupling passes take candidates by the wavefront (the spheres around 64
SPH particles staged together, a sphere's SPH candidates 64 at a time over the
column bounds): against the oracle on identical state, with one sphere and with
numbers around a group's, with all spheres in one corner across the periodic
faces (several rounds of 64 spheres a group), with coupling radii of several
sphere cells, uneven h, and in the closed box.  Bound: the passes' 1e-12."""
import numpy as np
import pytest

import oracle
import sphdem as sd

pytestmark = pytest.mark.gpu


def normwise(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


def corner(n_dem, spread):
    c = sd.sediment_case(nf=12, n_dem=n_dem, seed=9)
    dem = np.flatnonzero(c.iam == sd.DEM)
    rng = np.random.default_rng(3)
    p = rng.normal(scale=spread, size=(len(dem), 3))
    p[:, 2] = np.abs(p[:, 2]) + 0.3
    p[:, :2] = np.mod(p[:, :2], 1.0)
    c.r[dem] = p
    return c


def radius(ratio):
    c = sd.sediment_case(nf=12, n_dem=90, seed=5)
    c.params.dem_search_radius = c.params.coupling_radius / ratio
    c.h[c.iam == sd.DEM] = c.params.dem_search_radius
    return c


def uneven():
    c = sd.sediment_case(nf=16, nz=12, n_dem=80, seed=6)
    sph = np.isin(c.iam, (sd.SPH, sd.SPH_BOUNDARY))
    c.h[sph] *= 1.0 - 0.3 * np.random.default_rng(2).random(sph.sum())
    return c


CASES = {"one": lambda: sd.sediment_case(nf=12, n_dem=1, seed=1),
         "three": lambda: sd.sediment_case(nf=10, nz=12, n_dem=3, seed=2),
         "many": lambda: sd.sediment_case(nf=14, nz=12, n_dem=300, seed=3),
         "corner65": lambda: corner(65, 0.02), "corner300": lambda: corner(300, 0.06),
         "radius4": lambda: radius(4.0), "radius16": lambda: radius(16.0), "uneven": uneven,
         "closed": lambda: sd.dambreak_case(nf=12, with_dem=100, liq_dem_flags=True)}


@pytest.mark.parametrize("name", sorted(CASES))
def test_coupling_passes_against_the_oracle(name):
    c = CASES[name]()
    sim, orc = sd.Sim(c), oracle.Oracle(c)
    rng = np.random.default_rng(7)
    fd = np.zeros((c.n, 3))
    dem = c.iam == sd.DEM
    sph = np.isin(c.iam, (sd.SPH, sd.SPH_BOUNDARY))
    fd[dem] = rng.normal(size=(dem.sum(), 3)) * 1e-3
    vh = rng.normal(size=(c.n, 3)) * 0.05
    for x in (sim, orc):
        x.set("fdrag", fd)
        x.set("vhat", vh)
    orc.refresh_ghosts()
    sim.pass_("porosity")
    orc.pass_("porosity")
    assert normwise(sim.get("shepSum")[dem], orc.get("shepSum")[dem]) < 1e-12
    for nm in ("porosity", "fdrag", "f"):
        assert normwise(sim.get(nm)[sph], orc.get(nm)[sph]) < 1e-12, nm
    for nm in ("f", "fp", "fv", "fb"):
        x = rng.normal(size=(c.n, 3))
        sim.set(nm, x)
        orc.set(nm, x)
    orc.refresh_ghosts()
    sim.pass_("fpi")
    orc.pass_("fpi")
    for nm in ("fdrag", "fvel", "porosity", "shepSum", "fb", "fv"):
        assert normwise(sim.get(nm)[dem], orc.get(nm)[dem]) < 1e-12, nm
    sim.close()
