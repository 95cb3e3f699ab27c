"""Fields read into the caller's memory: sizes below and above the one from
which a context's helper threads take part (4 MiB), whole and partial last
pieces, into aligned and odd addresses, and two contexts read by two threads at
once: the values that were set."""
import ctypes
import threading

import numpy as np
import pytest

import sphdem as sd

pytestmark = pytest.mark.gpu


def roundtrip(sim, n, seed):
    rng = np.random.default_rng(seed)
    for name, shape in (("f", (n, 3)), ("press", (n,))):
        x = rng.random(shape)
        sim.set(name, x)
        assert np.array_equal(sim.get(name), x), name
        raw = np.zeros(x.nbytes + 16, np.uint8)  # an odd address, and what follows it
        raw[-9:] = 7
        at = raw.ctypes.data + 7
        sim._check(sim.lib.sphdem_get_field(sim.ctx, sd.FIELD[name], ctypes.c_void_p(at)))
        assert raw[7:7 + x.nbytes].tobytes() == x.tobytes(), name
        assert (raw[-9:] == 7).all() and (raw[:7] == 0).all()


@pytest.mark.parametrize("nf", [8, 43, 45, 47, 60, 72])
def test_sizes_on_both_sides_of_the_helpers(nf):
    case = sd.dambreak_case(nf=nf, dx=0.32 / nf)
    sim = sd.Sim(case)
    roundtrip(sim, case.n, nf)
    t = sim.get("iam")
    there = t != 255  # a coarse lattice's outer walls lie outside the domain
    assert there.any() and np.array_equal(t[there], case.iam[there])
    sim.close()


def test_two_contexts_read_at_once():
    cases = [sd.dambreak_case(nf=nf, dx=0.32 / nf) for nf in (52, 56)]
    sims = [sd.Sim(c) for c in cases]
    failed = []

    def work(k):
        try:
            for i in range(4):
                roundtrip(sims[k], cases[k].n, 10 * k + i)
        except BaseException as e:  # noqa: BLE001 -- reported by the test's thread
            failed.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for s in sims:
        s.close()
