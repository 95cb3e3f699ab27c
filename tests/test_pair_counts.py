"""Pair searches: more targets than one tile of scanned tiles holds (16,777,216)
hand out their pairs, as the list build does; and a search that only counts takes
no memory for the pairs."""
import ctypes

import numpy as np
import pytest
import torch

import sphdem as sd

pytestmark = pytest.mark.gpu


def test_more_targets_than_a_tile_of_tiles():
    N, dx = 257, 0.01  # a lattice of 16,974,593 targets, radius 1.2 dx: six neighbours inside
    c = sd.dambreak_case(nf=4, dx=dx)
    P = c.params
    for k in range(3):
        P.rmin[k], P.rmax[k] = 0.0, N * dx
        P.proc_domain[2 * k], P.proc_domain[2 * k + 1] = 0.0, N * dx
    x = (np.arange(N) + 0.5) * dx
    r = np.stack(np.meshgrid(x, x, x, indexing="ij"), axis=-1).reshape(-1, 3)
    n = len(r)
    z = np.zeros((n, 3))
    case = sd.Case("lattice", P, r, z, z, np.full(n, dx ** 3 * 1000.0), np.full(n, 0.6 * dx),
                   np.full(n, 1000.0), np.full(n, sd.SPH, np.int32), sd.HOOKS_NONE, {})
    print("lattice of", n, flush=True)
    sim = sd.Sim(case)
    sim.reset()
    want = 6 * N * N * (N - 1)
    assert sim.pair_count(sd.PAIRS_SPH) == want
    a, b, im = (torch.empty(want, dtype=torch.int32, device="cuda") for _ in range(3))
    cnt = ctypes.c_int64()
    torch.cuda.synchronize()
    assert sim.lib.sphdem_get_pairs_device(sim.ctx, sd.PAIRS_SPH, ctypes.byref(cnt), a.data_ptr(),
                                           b.data_ptr(), im.data_ptr(), want) == 0
    assert cnt.value == want
    per = torch.bincount(a.long(), minlength=n)
    edge = torch.zeros(N, dtype=torch.int64, device="cuda")
    edge[[0, -1]] = 1  # faces a lattice index lies on
    on = edge[:, None, None] + edge[None, :, None] + edge[None, None, :]
    assert torch.equal(per, 6 - on.reshape(-1))
    step = (a - b).abs()
    assert bool(((step == 1) | (step == N) | (step == N * N)).all())
    assert bool((im == 13).all())
    sim.close()


def test_a_count_keeps_no_pairs():
    """The room for pairs kept between the count and the write (128 a query) is
    taken by a search that writes."""
    sim = sd.Sim(sd.sediment_case(nf=32, n_dem=64, seed=1))
    sim.reset()
    sim.pair_count(sd.PAIRS_DEM2SPH)
    torch.cuda.synchronize()
    kept = 4 * 128 * sim.case.n
    before = torch.cuda.mem_get_info()[0]
    cnt = sim.pair_count(sd.PAIRS_SPH2DEM)
    assert before - torch.cuda.mem_get_info()[0] < kept // 4  # counts and offsets
    assert len(sim.pairs(sd.PAIRS_SPH2DEM)) == cnt
    sim.close()
