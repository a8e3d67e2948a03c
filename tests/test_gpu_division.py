"""The quotients of the FP64 psi sweeps, formed from a reciprocal, are those of
a division. With spacings so wide that the neighbours' terms vanish (1 / dx^2
= 0) one sweep is psi / (1 + dt (|psi|^2 - eps)), compared with numpy's to
the bit on 1e6 values of any size whose remainder does not underflow (from
2^-900 on; below 2^-960 it may, and the last bit with it)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
nat = pytest.importorskip("svirl_amd._native")


@pytest.fixture(scope="module", autouse=True)
def _init():
    nat.init(0)


@pytest.mark.parametrize("wg", [0, 8])  # register tiles, row-marching
@pytest.mark.parametrize("wide", [False, True])
def test_quotients_are_those_of_a_division(wg, wide):
    Nx, Ny, dt = 900, 560, 0.1
    rng = np.random.default_rng(11)
    n = Nx * Ny
    e = rng.integers(-900, 400, size=(2, n)) if wide else rng.integers(-4, 3, size=(2, n))
    v = np.ldexp(rng.choice([-1.0, 1.0], size=(2, n)) * (1.0 + rng.random((2, n))), e)
    psi = v[0] + 1j * v[1]
    up = nat.DeviceArray.from_host
    nab = (Nx - 1) * Ny + Nx * (Ny - 1)
    P = [up(psi)] + [nat.DeviceArray.zeros(n, psi.dtype) for _ in range(2)]
    Q = [nat.DeviceArray.zeros(nab, np.float64) for _ in range(3)]
    Pp = (ctypes.c_void_p * 3)(*[b.ptr for b in P])
    Qp = (ctypes.c_void_p * 3)(*[b.ptr for b in Q])
    pc, qc = ctypes.c_int32(0), ctypes.c_int32(0)
    prm = nat.TDParams()
    prm.dt, prm.eps, prm.stop_psi, prm.stop_A = dt, 1.0, 1e-6, 1e-6
    prm.rand_t, prm.max_sweeps = 1, 1
    sw = (ctypes.c_int32 * 2)()
    nat.call("glx_td_run", nat.GLX_F64, nat.Grid(Nx, Ny, 1e200, 1e200), ctypes.byref(prm), None, None, Pp,
             ctypes.byref(pc), Qp, ctypes.byref(qc), None, None, 1, sw, wg, 256)
    assert sw[0] == 1
    den = 1.0 + dt * (v[0] * v[0] + v[1] * v[1] - 1.0)
    out = P[pc.value].get()
    assert np.array_equal(out.real, v[0] / den) and np.array_equal(out.imag, v[1] / den)
