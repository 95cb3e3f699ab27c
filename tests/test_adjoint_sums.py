"""The parameter sums of the adjoint's backward passes (viscosity, drag_a,
drag_b) over many queries: against the exact sum (fsum) of the contributions
that the same kernels give for each query by itself.

The bound: a workgroup of 256 queries may round its running total once, M = N /
256 roundings in all, in an order that varies.  With terms of one sign the total
grows evenly and M roundings of up to half a unit in the last place of it leave
an rms error of sqrt(M / 36) such units (each uniform over a unit of a total k/M
of the last: the mean of k^2/M^2 is 1/3, of a uniform square 1/12).  Three times
that is allowed."""
import ctypes
import math

import numpy as np
import pytest
import torch

import sphdem as sd
import sphdem_adjoint as sa

pytestmark = pytest.mark.gpu


def consts():
    c = sa.AdjConsts(wcon=21.0 / (256.0 * math.pi), viscosity=1e-3, dens=1000.0, pi=math.pi,
                     dem_radius=0.05, dem_vol=4.0 / 3.0 * math.pi * 0.05 ** 3, drag_a=3.7,
                     drag_b=0.65)
    return c


def bound(total, queries):
    return 3.0 * math.sqrt(max(queries / 256.0, 1.0) / 36.0) * np.spacing(abs(total))


def sums(call, n, params):
    """(the call's sums over all queries, the exact sums of those of each alone)"""
    lib = sa._adj_lib()
    one = torch.zeros((n, 5), dtype=torch.float64, device="cuda")
    for i in range(n):
        call(lib, i, 1, one[i])
    each = one.cpu().numpy()
    whole = []
    for _ in range(4):  # their order varies
        p = torch.zeros(5, dtype=torch.float64, device="cuda")
        call(lib, 0, n, p)
        whole.append(p.cpu().numpy())
    exact = np.array([math.fsum(each[:, k]) for k in range(5)])
    for k in params:
        assert np.all(each[:, k] >= 0) or np.all(each[:, k] <= 0)
        assert abs(exact[k]) > 0
        worst = max(abs(w[k] - exact[k]) for w in whole)
        assert worst <= bound(exact[k], n), (k, worst / np.spacing(abs(exact[k])))


def dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device="cuda")


def stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("n", [1 << 17, 5003])
def test_drag_on_spheres(n):
    """n spheres, each over the same eight fluid particles, their velocities and
    the adjoints of their drag different."""
    rng = np.random.default_rng(n)
    m = 8
    tot = m + n
    r = np.concatenate([0.05 * rng.random((m, 3)), 0.05 * rng.random((n, 3))])
    vh = np.concatenate([np.zeros((m, 3)), 0.5 + rng.random((n, 3))])
    f = dict(r=dev(r), vhat=dev(vh), h=dev(np.full(tot, 0.1)), dens=dev(np.full(tot, 1000.0)),
             mass=dev(np.concatenate([np.full(m, 1000.0 * 0.1 ** 3), np.full(n, 1.3)])),
             fpfb=dev(np.zeros((tot, 3))), fv=dev(np.zeros((tot, 3))),
             por=dev(np.full(tot, 0.8)))
    q = dev(np.arange(m, tot), torch.int32)
    off = dev(np.arange(n + 1) * m, torch.int64)
    b = dev(np.tile(np.arange(m), n), torch.int32)
    img = dev(np.full(n * m, 13), torch.int32)
    gf = dev(-vh * (0.5 + rng.random((tot, 1))))  # along the slip: every term of one sign
    out = {k: torch.zeros_like(f[k]) for k in ("r", "vhat", "h", "dens", "fpfb", "fv", "por")}
    c = consts()
    fl = sa.AdjFields(**{k: v.data_ptr() for k, v in f.items()})

    def call(lib, first, count, params):
        g = sa.AdjGrads(params=params.data_ptr(), **{k: v.data_ptr() for k, v in out.items()})
        rc = lib.sphdem_adj_fpi_bwd(count, q.data_ptr() + 4 * first, off.data_ptr() + 8 * first,
                                    sa._ptr(b), sa._ptr(img), ctypes.byref(fl), ctypes.byref(c),
                                    sa._ptr(gf), ctypes.byref(g), stream())
        assert rc == 0

    sums(call, n, (1, 2))


@pytest.mark.parametrize("n", [1 << 17, 5003])
def test_viscous_force(n):
    """n particles in pairs by themselves; the adjoint of the viscous force along
    it."""
    n &= ~1
    rng = np.random.default_rng(n)
    r = np.repeat(rng.random((n // 2, 3)), 2, axis=0)
    r[1::2] += 0.02 + 0.02 * rng.random((n // 2, 3))
    vh = rng.normal(size=(n, 3))
    f = dict(r=dev(r), vhat=dev(vh), h=dev(np.full(n, 0.05)), dens=dev(np.full(n, 1000.0)),
             mass=dev(np.full(n, 0.3)), omega=dev(np.ones(n)), pdr2=dev(np.full(n, 1e-3)),
             iam=dev(np.full(n, sd.SPH), torch.int32))
    other = np.arange(n) ^ 1
    q = dev(np.arange(n), torch.int32)
    off = dev(np.arange(n + 1), torch.int64)
    b = dev(other, torch.int32)
    img = dev(np.full(n, 13), torch.int32)
    gv = dev(vh[other] - vh)
    gp = dev(np.zeros((n, 3)))
    out = {k: torch.zeros_like(f[k]) for k in ("r", "vhat", "h", "dens", "omega", "pdr2")}
    c = consts()
    fl = sa.AdjFields(**{k: v.data_ptr() for k, v in f.items()})

    def call(lib, first, count, params):
        g = sa.AdjGrads(params=params.data_ptr(), **{k: v.data_ptr() for k, v in out.items()})
        rc = lib.sphdem_adj_force_bwd(count, q.data_ptr() + 4 * first, off.data_ptr() + 8 * first,
                                      sa._ptr(b), sa._ptr(img), ctypes.byref(fl),
                                      ctypes.byref(c), sa._ptr(gv), sa._ptr(gp), ctypes.byref(g),
                                      stream())
        assert rc == 0

    sums(call, n, (0,))


def test_launches_beside_and_behind_one_another():
    """More launches in flight than hold partial sums of their own, on several
    streams and without a wait, and one replayed from a graph: each result is its
    own launch's."""
    n, m = 4096, 8
    rng = np.random.default_rng(2)
    r = np.concatenate([0.05 * rng.random((m, 3)), 0.05 * rng.random((n, 3))])
    vh = np.concatenate([np.zeros((m, 3)), 0.5 + rng.random((n, 3))])
    tot = m + n
    f = dict(r=dev(r), vhat=dev(vh), h=dev(np.full(tot, 0.1)), dens=dev(np.full(tot, 1000.0)),
             mass=dev(np.concatenate([np.full(m, 1.0), np.full(n, 1.3)])),
             fpfb=dev(np.zeros((tot, 3))), fv=dev(np.zeros((tot, 3))), por=dev(np.full(tot, 0.8)))
    q = dev(np.arange(m, tot), torch.int32)
    off = dev(np.arange(n + 1) * m, torch.int64)
    b = dev(np.tile(np.arange(m), n), torch.int32)
    img = dev(np.full(n * m, 13), torch.int32)
    gf = dev(-vh)
    out = {k: torch.zeros_like(f[k]) for k in ("r", "vhat", "h", "dens", "fpfb", "fv", "por")}
    c = consts()
    fl = sa.AdjFields(**{k: v.data_ptr() for k, v in f.items()})
    lib = sa._adj_lib()

    def launch(count, params):
        g = sa.AdjGrads(params=params.data_ptr(), **{k: v.data_ptr() for k, v in out.items()})
        assert lib.sphdem_adj_fpi_bwd(count, sa._ptr(q), sa._ptr(off), sa._ptr(b), sa._ptr(img),
                                      ctypes.byref(fl), ctypes.byref(c), sa._ptr(gf),
                                      ctypes.byref(g), stream()) == 0

    counts = [n, n // 3, n // 7, 5, 1]
    want = torch.zeros((len(counts), 5), dtype=torch.float64, device="cuda")
    for k, cnt in enumerate(counts):
        launch(cnt, want[k])
        torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    got = torch.zeros((600, 5), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    for i in range(len(got)):
        with torch.cuda.stream(streams[i % 3]):
            launch(counts[i % len(counts)], got[i])
    torch.cuda.synchronize()
    replayed = torch.zeros(5, dtype=torch.float64, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch(n, replayed)
    for i in range(3):
        replayed.zero_()
        graph.replay()
        launch(n, got[0].zero_())  # beside it, on another stream
        torch.cuda.synchronize()
        assert torch.allclose(replayed, want[0], rtol=1e-13, atol=0.0)
        assert torch.allclose(got[0], want[0], rtol=1e-13, atol=0.0)
    for i in range(len(got)):
        assert torch.allclose(got[i], want[i % len(counts)], rtol=1e-13, atol=0.0), i
