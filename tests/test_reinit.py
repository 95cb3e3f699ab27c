"""A density re-initialisation's ten iterations in the mixed form (one pass, then
a kernel in which each particle iterates over its kept distances) against ten
density passes: density and h bit for bit, over lists that fit the kept
distances and longer ones, neighbours of one mass and of several, numbers of
targets around a wavefront's and a workgroup's, and with periodic ghosts."""
import numpy as np
import pytest

import sphdem as sd

pytestmark = pytest.mark.gpu


def squeezed(by):
    def make():
        c = sd.dambreak_case(nf=12)
        m = c.r.mean(axis=0)
        c.r[:] = m + by * (c.r - m)
        return c
    return make


def masses():
    c = sd.dambreak_case(nf=12)
    c.mass[::3] *= 1.25
    return c


CASES = {"nf5": lambda: sd.dambreak_case(nf=5), "nf12": lambda: sd.dambreak_case(nf=12),
         "nf21": lambda: sd.dambreak_case(nf=21), "longer lists": squeezed(0.9),
         "longest lists": squeezed(0.82), "masses": masses,
         "ghosts": lambda: sd.sediment_case(nf=12, n_dem=20)}


@pytest.mark.parametrize("name", sorted(CASES))
def test_ten_iterations_equal_ten_passes(name):
    a, b = CASES[name](), CASES[name]()
    a.params.reinit_every, b.params.reinit_every = 1, 1 << 30
    one, ten = sd.Sim(a, precision=sd.MIXED), sd.Sim(b, precision=sd.MIXED)
    for x in (one, ten):
        g = x.globals()
        g.sphStep = 7  # a step that only the first re-initialises on
        x.set_globals(g)
        x.start()
    ten.reset()
    for _ in range(10):
        ten.pass_("density")
    before = np.asarray(b.dens)
    assert np.array_equal(one.get("dens"), ten.get("dens"))
    assert np.array_equal(one.get("h"), ten.get("h"))
    assert not np.array_equal(one.get("dens"), before)
    one.close()
    ten.close()
