"""B, J and J_s in column order (glx_bulk_observables_cols) against the row
order of glx_bulk_observables, to the bit, at sizes around its tile of 32 x
32 nodes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
nat = pytest.importorskip("svirl_amd._native")


@pytest.fixture(scope="module", autouse=True)
def _init():
    nat.init(0)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shape", [(4, 4), (32, 33), (33, 32), (5, 130), (100, 65)])
@pytest.mark.parametrize("abei", [True, False])
def test_column_order_equals_row_order(dtype, shape, abei):
    Nx, Ny = shape
    rng = np.random.default_rng(Nx + 7 * Ny)
    Na, Nb, Nc = (Nx - 1) * Ny, Nx * (Ny - 1), (Nx - 1) * (Ny - 1)
    up = nat.DeviceArray.from_host
    psi = (rng.normal(size=Nx * Ny) + 1j * rng.normal(size=Nx * Ny)).astype(np.complex64 if dtype == np.float32 else complex)
    d_psi, d_ab = up(psi), up(rng.normal(size=Na + Nb).astype(dtype))
    d_ae = up(rng.normal(size=Na + Nb).astype(dtype)) if abei else None
    d_mt = up((rng.random(Nc) > 0.2).astype(np.uint8))
    outs = []
    for name in ("glx_bulk_observables", "glx_bulk_observables_cols"):
        B, J, S = (nat.DeviceArray.zeros(n, dtype) for n in (Nc, Na + Nb, Na + Nb))
        nat.call(name, nat.prec_of(dtype), nat.Grid(Nx, Ny, 0.5, 0.4), 16.0, 0.2, d_mt.ptr, d_psi.ptr, nat.ptr(d_ae),
                 d_ab.ptr, B.ptr, J.ptr, S.ptr)
        outs.append((B.get(), J.get(), S.get()))
    (B0, J0, S0), (B1, J1, S1) = outs
    assert np.array_equal(B1.reshape(Nx - 1, Ny - 1), B0.reshape(Ny - 1, Nx - 1).T)
    for v0, v1 in ((J0, J1), (S0, S1)):
        assert np.array_equal(v1[:Na].reshape(Nx - 1, Ny), v0[:Na].reshape(Ny, Nx - 1).T)
        assert np.array_equal(v1[Na:].reshape(Nx, Ny - 1), v0[Na:].reshape(Ny - 1, Nx).T)
    # one output alone
    J = nat.DeviceArray.zeros(Na + Nb, dtype)
    nat.call("glx_bulk_observables_cols", nat.prec_of(dtype), nat.Grid(Nx, Ny, 0.5, 0.4), 16.0, 0.2, None, None,
             nat.ptr(d_ae), d_ab.ptr, None, J.ptr, None)
    assert np.array_equal(J.get(), J1)
