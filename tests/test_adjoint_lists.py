"""The pair passes' kernels take a query's list by a group of lanes: forward and
backward over lists of every length around a group's and a wavefront's (empty
ones and one entry, one more and one less than a group, several rounds) equal
torch autograd of the same passes.  Particles sit in clusters, every ordered
pair of a cluster's in the sets; bounds as for the physical case (1e-12 of the
largest value forward, 1e-10 backward, 1e-9 the parameters)."""
import numpy as np
import pytest
import torch

import sphdem as sd
import sphdem_adjoint as sa
from adjoint_ref import TorchPasses

pytestmark = pytest.mark.gpu


def normwise(a, b):
    return float((a - b).abs().max() / max(float(b.abs().max()), 1e-300))


def clusters(sph_sizes, dem_sizes, seed):
    """(model, positions, pair sets): cluster k holds sph_sizes[k] SPH-group
    particles and dem_sizes[k] spheres within a ball of radius h."""
    case = sd.adjoint_case(nf=12, nz=12, n_dem=max(sum(dem_sizes), 1), seed=7)
    rng = np.random.default_rng(seed)
    sph = rng.permutation(np.flatnonzero(np.isin(case.iam, (sd.SPH, sd.SPH_BOUNDARY))))
    dem = np.flatnonzero(case.iam == sd.DEM)
    h = case.params.h
    sets = {sd.PAIRS_SPH: [], sd.PAIRS_SPH2DEM: [], sd.PAIRS_DEM2SPH: []}
    r = case.r.copy()
    i = j = 0
    for ns, nd in zip(sph_sizes, dem_sizes):
        S, D = sph[i:i + ns], dem[j:j + nd]
        i, j = i + ns, j + nd
        both = np.concatenate([S, D])
        d = rng.normal(size=(len(both), 3))
        d *= (h * rng.random(len(both)) ** (1 / 3) / np.linalg.norm(d, axis=1))[:, None]
        r[both] = rng.uniform(0.3, 0.7, 3) * [1.0, 1.0, 0.5] + d
        for kind, A, B in ((sd.PAIRS_SPH, S, S), (sd.PAIRS_SPH2DEM, S, D),
                           (sd.PAIRS_DEM2SPH, D, S)):
            sets[kind] += [(a, b, 13) for a in A for b in B if a != b]
    case.r = r
    # particles under no case's order: identity keeps the indices
    model = sa.StepModel(case, device="cuda", passes=TorchPasses(), pairs=None)
    place = np.empty(case.n, np.int64)
    where = model.original(torch.arange(case.n, device="cuda", dtype=torch.float64))
    place[:] = where.cpu().numpy().astype(np.int64)  # model index of an original one
    L = torch.as_tensor([1.0, 1.0, 1.0], dtype=torch.float64, device="cuda")
    ps = {}
    for kind, rows in sets.items():
        t = np.array(rows, np.int64).reshape(-1, 3)
        t[:, :2] = place[t[:, :2]]
        ps[kind] = sa.PairSet(torch.as_tensor(t, device="cuda"), case.n, L)
    S = model.initial_state()
    return model, S, ps


@pytest.mark.parametrize("sph_sizes, dem_sizes", [
    ((1, 2, 3, 8, 9, 10), (0, 1, 2, 7, 8, 9)),
    ((15, 16, 17, 18, 31, 33, 34), (1, 15, 16, 17, 3, 0, 25)),
    ((63, 64, 65, 66), (1, 1, 31, 33)),
    ((127, 128, 129, 130, 200), (2, 1, 5, 1, 1)),
    ((2,), (1,)),
])
def test_lists_of_every_length_around_a_group(sph_sizes, dem_sizes):
    model, S, ps = clusters(sph_sizes, dem_sizes, len(sph_sizes))
    th = model.params(requires_grad=True)
    C = sa._Ctx(model, th)
    gen = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda t: torch.rand(t.shape, generator=gen, dtype=t.dtype, device=t.device)
    r, h, dens = S["r"], S["h"], S["dens"] * 0.02  # fluid volumes that fill a sphere's sum
    h = torch.where(model.grp, h * (1.0 + 0.1 * rnd(h)), h)
    vhat = rnd(r) - 0.5
    omega, por, pdr2 = 0.9 + 0.2 * rnd(h), 0.5 + 0.4 * rnd(h), 1e-3 * rnd(h)
    fp, fv, fdrag = rnd(r) - 0.5, rnd(r) - 0.5, rnd(r) - 0.5
    cases = {
        "omega": (lambda P, x: P.omega(C, ps[sd.PAIRS_SPH], *x), [r, h, dens], []),
        "dddt": (lambda P, x: P.dddt(C, ps[sd.PAIRS_SPH], *x), [r, vhat, h, omega], []),
        "force": (lambda P, x: P.force(C, ps[sd.PAIRS_SPH], *x, th["viscosity"]),
                  [r, vhat, h, dens, omega, pdr2], ["viscosity"]),
        "coupling": (lambda P, x: P.coupling(C, ps[sd.PAIRS_SPH2DEM], *x), [r, dens, fdrag], []),
        "fpi": (lambda P, x: P.fpi(C, ps[sd.PAIRS_DEM2SPH], *x, th["viscosity"], th["drag_a"],
                                   th["drag_b"]),
                [r, vhat, h, dens, fp, fv, por], ["viscosity", "drag_a", "drag_b"]),
    }
    for name, (fn, xs, pnames) in cases.items():
        out = {}
        for tag, P in (("hip", sa.HipPasses()), ("torch", TorchPasses())):
            x = [t.detach().clone().contiguous().requires_grad_(True) for t in xs]
            for k in pnames:
                th[k].grad = None
            y = fn(P, x)
            y = y if isinstance(y, tuple) else (y,)
            torch.autograd.backward(y, [torch.sin(7.0 * torch.arange(
                t.numel(), device=t.device, dtype=t.dtype)).reshape(t.shape) for t in y])
            zero = [torch.zeros_like(t) for t in x]
            out[tag] = ([t.detach() for t in y],
                        [z if t.grad is None else t.grad for t, z in zip(x, zero)],
                        [float(th[k].grad) for k in pnames])
        (yh, gh, ph), (yt, gt, pt) = out["hip"], out["torch"]
        for a, b in zip(yh, yt):
            assert normwise(a, b) < 1e-12, name
        for i, (a, b) in enumerate(zip(gh, gt)):
            assert normwise(a, b) < 1e-10, (name, i)
        for k, a, b in zip(pnames, ph, pt):
            assert a == pytest.approx(b, rel=1e-9, abs=1e-300), (name, k)
