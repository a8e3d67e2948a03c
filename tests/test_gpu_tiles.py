"""Time-dependent runs on register tiles (the default of glx_td_run where a
grid fits them) against the row-marching solves (an explicit workgroup
count): FP64 fields and sweep counts to the bit, FP32 to its rounding. Sizes
at and around the tiles' edges and for each tile shape; runs whose solves
are redone from an earlier sweep, need more than 32 sweeps, or stop at the
sweep limit (FP64, where the schedule shows to the bit)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
nat = pytest.importorskip("svirl_amd._native")


H = 0.1


@pytest.fixture(scope="module", autouse=True)
def _init():
    nat.init(0)


def state(Nx, Ny, dtype, disorder, seed):
    rng = np.random.default_rng(seed)
    cd = np.complex64 if dtype == np.float32 else np.complex128
    psi = (rng.random(Nx * Ny) * np.exp(2j * np.pi * rng.random(Nx * Ny))).astype(cd)
    # the gauge of the field plus noise: FP32 resolves the stop criterion of
    # 1e-6 only in what is left of A when that gauge is taken out
    a = -0.5 * H * (np.arange(Ny) * 0.5 - 0.25 * (Ny - 1))[:, None] + np.zeros((Ny, Nx - 1))
    b = 0.5 * H * (np.arange(Nx) * 0.5 - 0.25 * (Nx - 1))[None, :] + np.zeros((Ny - 1, Nx))
    ab = np.concatenate([a.ravel(), b.ravel()])
    ab = (ab + 0.3 * rng.standard_normal(ab.size)).astype(dtype)
    mt = (rng.random((Nx - 1) * (Ny - 1)) > 0.15).astype(np.uint8) if disorder else None
    eps = (1.0 + 0.2 * rng.standard_normal(Nx * Ny)).astype(dtype) if disorder else None
    return psi, ab, mt, eps


def run(Nx, Ny, dtype, fields, kappa, wg, nsteps, dt=0.1, sigma=200.0, max_sweeps=1024, eqn=0):
    psi, ab, mt, eps = fields
    up = nat.DeviceArray.from_host
    P = [up(psi)] + [nat.DeviceArray.zeros(psi.size, psi.dtype) for _ in range(2)]
    Q = [up(ab)] + [nat.DeviceArray.zeros(ab.size, ab.dtype) for _ in range(2)]
    Pp = (ctypes.c_void_p * 3)(*[b.ptr for b in P])
    Qp = (ctypes.c_void_p * 3)(*[b.ptr for b in Q])
    pc, qc = ctypes.c_int32(0), ctypes.c_int32(0)
    d_mt, d_eps = (None if v is None else up(v) for v in (mt, eps))
    prm = nat.TDParams()
    prm.dt, prm.eps, prm.kappa2, prm.rho, prm.H = dt, 0.0 if eps is not None else 1.0, kappa * kappa, 1.0 / sigma, H
    prm.stop_psi = prm.stop_A = 1e-6
    prm.rand_t, prm.solveA, prm.max_sweeps, prm.eqn = 1, 1 if kappa else 0, max_sweeps, eqn
    sw = (ctypes.c_int32 * (2 * nsteps))()
    nat.call("glx_td_run", nat.prec_of(dtype), nat.Grid(Nx, Ny, 0.5, 0.5), ctypes.byref(prm), nat.ptr(d_eps),
             nat.ptr(d_mt), Pp, ctypes.byref(pc), Qp, ctypes.byref(qc), None, None, nsteps, sw, wg, 256)
    return P[pc.value].get(), Q[qc.value].get(), np.frombuffer(sw, dtype=np.int32).reshape(nsteps, 2).copy()


def compare(Nx, Ny, dtype, kappa, disorder, nsteps, **kw):
    f = state(Nx, Ny, dtype, disorder, seed=Nx * 7 + Ny)
    psi, ab, sw = run(Nx, Ny, dtype, f, kappa, 0, nsteps, **kw)
    psi1, ab1, sw1 = run(Nx, Ny, dtype, f, kappa, 8, nsteps, **kw)
    assert np.all(np.isfinite(psi1.view(dtype))) and sw1[:, 0].min() > 0
    if dtype == np.float64:
        assert np.array_equal(sw, sw1)
        assert np.array_equal(psi, psi1) and np.array_equal(ab, ab1)
    else:
        # a sweep's rounding (6e-8 of values up to 2, A less its gauge part)
        # over the sweeps of a few steps; a stop rule of 1e-6 met one sweep apart
        assert np.all(np.abs(sw - sw1) <= 1)
        assert np.max(np.abs(psi - psi1)) <= 2e-5
        assert np.max(np.abs(ab - ab1)) <= 2e-5


# smallest grids; one tile exactly, one node more, several tiles and a
# remainder; one grid per larger tile shape
SIZES = [(4, 4), (5, 33), (56, 8), (57, 9), (113, 25), (64, 200), (300, 520), (530, 410), (701, 690), (771, 1283)]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("kappa", [0.0, 5.0])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_tiles_equal_rows(size, kappa, dtype):
    compare(*size, dtype, kappa, disorder=(size[0] + size[1]) % 2 == 1, nsteps=3)


@pytest.mark.parametrize("dt,sigma,max_sweeps,eqn", [
    (0.02, 50.0, 1024, 0),   # A sweep counts that fall and rise
    (0.8, 400.0, 1024, 0),   # more than 32 psi sweeps a step
    (0.1, 200.0, 3, 0),      # the sweep limit, odd
    (0.1, 200.0, 17, 0),
    (0.1, 200.0, 1024, 1),   # psi only, A present
])
def test_tile_schedules_equal_rows(dt, sigma, max_sweeps, eqn):
    compare(150, 131, np.float64, 5.0, True, 6, dt=dt, sigma=sigma, max_sweeps=max_sweeps, eqn=eqn)


@pytest.mark.parametrize("kappa", [0.0, 5.0])
@pytest.mark.parametrize("size", [(129, 129), (129, 513), (257, 65), (513, 257), (701, 690)])
def test_fp32_tiles_stop_where_fp64_does(size, kappa):
    # the FP32 tiles carry the changes themselves, to 1e-7 of their size, so
    # the stop rule is met at the sweep where 64-bit iterates meet it (the
    # difference of two FP32 iterates is off by up to 1e-1 of the rule)
    f = state(*size, np.float32, True, seed=size[0] + 3 * size[1])
    f64 = (f[0].astype(np.complex128), f[1].astype(np.float64), f[2], f[3].astype(np.float64))
    sw = run(*size, np.float32, f, kappa, 0, 10)[2]
    sw64 = run(*size, np.float64, f64, kappa, 8, 10)[2]
    assert np.array_equal(sw[:, 0], sw64[:, 0])


def run_batch(insts, dtype, nsteps, noalloc):
    """[(Nx, Ny, kappa, fields)] advanced together; (psi, ab, sweeps) of each."""
    up = nat.DeviceArray.from_host
    arr = (nat.BatchInstance * len(insts))()
    bufs = []
    for I, (Nx, Ny, kappa, (psi, ab, mt, eps)) in zip(arr, insts):
        P = [up(psi)] + [nat.DeviceArray.zeros(psi.size, psi.dtype) for _ in range(2)]
        Q = [up(ab)] + [nat.DeviceArray.zeros(ab.size, ab.dtype) for _ in range(2)]
        d_mt, d_eps = (None if v is None else up(v) for v in (mt, eps))
        bufs.append((P, Q, d_mt, d_eps))
        I.g = nat.Grid(Nx, Ny, 0.5, 0.5)
        prm = I.p
        prm.dt, prm.eps, prm.kappa2, prm.rho, prm.H = 0.1, 0.0 if eps is not None else 1.0, kappa * kappa, 0.005, H
        prm.stop_psi = prm.stop_A = 1e-6
        prm.rand_t, prm.solveA, prm.max_sweeps, prm.eqn = 1, 1 if kappa else 0, 1024, 0
        I.eps_map, I.mt = nat.ptr(d_eps), nat.ptr(d_mt)
        for j in range(3):
            I.psi[j], I.ab[j] = P[j].ptr, Q[j].ptr
        I.psi_cur = I.ab_cur = 0
    n = len(insts)
    sw = (ctypes.c_int32 * (2 * n * nsteps))()
    if noalloc:
        nat.call("glx_batch_td_run_noalloc", nat.prec_of(dtype), arr, n, nsteps, sw, 0, 0, None, 0)
    else:
        nat.call("glx_batch_td_run", nat.prec_of(dtype), arr, n, nsteps, sw, 0, 0, 0, None, 0)
    sw = np.frombuffer(sw, dtype=np.int32).reshape(nsteps, n, 2)
    return [(b[0][I.psi_cur].get(), b[1][I.ab_cur].get(), sw[:, k].copy()) for k, (I, b) in enumerate(zip(arr, bufs))]


# one instance; many small ones, with and without A; more tiles than one
# launch holds; one grid that no tile shape holds among ones that fit
BATCHES = [[(57, 9)], [(4, 4), (33, 70), (130, 65), (56, 24), (5, 300)] * 5, [(400, 500)] * 6 + [(65, 65)],
           [(1100, 1100), (129, 257), (1100, 1100), (64, 64)]]


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("batch", range(len(BATCHES)))
def test_batch_on_tiles_equals_rows(batch, noalloc):
    sizes = BATCHES[batch]
    insts = [(*s, 0.0 if k % 3 == 1 else 5.0, state(*s, np.float64, k % 2 == 0, seed=k)) for k, s in enumerate(sizes)]
    for (psi, ab, sw), (Nx, Ny, kappa, f) in zip(run_batch(insts, np.float64, 3, noalloc), insts):
        psi1, ab1, sw1 = run(Nx, Ny, np.float64, f, kappa, 8, 3)
        assert np.array_equal(sw, sw1)
        assert np.array_equal(psi, psi1) and np.array_equal(ab, ab1)
