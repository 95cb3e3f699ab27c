"""r or h set after a run, while the step's near lists are in place: what the exact
lists are made from is kept without new memory, and through a checkpoint saved in
between."""
import numpy as np
import pytest
import torch

import sphdem as sd

pytestmark = pytest.mark.gpu


def test_setting_h_after_a_run_takes_no_memory():
    sim = sd.Sim(sd.sediment_case(nf=64, n_dem=64, seed=1))
    sim.run(1)
    h = sim.get("h")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    sim.set("h", 0.9 * h)
    assert torch.cuda.mem_get_info()[0] == before
    sim.close()


@pytest.mark.parametrize("make", [lambda: sd.sediment_case(nf=13, nz=13, n_dem=40, seed=13),
                                  lambda: sd.dambreak_case(nf=12)])
def test_pairs_after_a_checkpoint_saved_in_between(make):
    got = []
    for seg in (64, 0):
        sim = sd.Sim(make())
        sim.set_tile_shape(seg, 256)
        sim.run(2)
        d = np.random.default_rng(4)
        r, h = sim.get("r"), sim.get("h")
        sim.set("r", r + 1e-3 * (d.random(r.shape) - 0.5))
        sim.set("h", h * (0.8 + 0.1 * d.random(h.shape)))
        blob = sim.checkpoint()
        pairs = sim.pairs(sd.PAIRS_SPH)
        sim.restore(blob)
        sim.run(1)
        got.append((pairs, sim.get("r"), sim.pairs(sd.PAIRS_SPH)))
        sim.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
