"""FP32 time steps on register tiles are as accurate as the row-marching ones
where a step shrinks psi: away from the middle of a large sample the vector
potential outgrows smooth vortices, and |psi| falls to a fourth and less in a
step. The error of 20 steps against 64 bits (same inputs, same sweeps) is the
sum of the roundings of 3e5 to 5e5 components, so the two forms' errors scatter by
less than a percent; in a tile the four links are summed in a chain where the
rows sum them in pairs, which is worth up to a tenth. Sums of changes from
the step's first sweep on gave 1.6 times the rows' error here."""
import numpy as np
import pytest
from scipy.ndimage import gaussian_filter

from tests.test_gpu_tiles import run, state

pytestmark = pytest.mark.gpu
nat = pytest.importorskip("svirl_amd._native")


@pytest.fixture(scope="module", autouse=True)
def _init():
    nat.init(0)


@pytest.mark.parametrize("kappa", [0.0, 5.0])
@pytest.mark.parametrize("size", [(513, 513), (385, 641)])
def test_fp32_error_is_that_of_rows(size, kappa):
    Nx, Ny = size
    rng = np.random.default_rng(Nx + Ny)
    z = gaussian_filter(rng.standard_normal((2, Ny, Nx)), (0, 4, 4), mode='wrap')
    z = (z[0] + 1j * z[1]) / z[0].std()
    psi = (z / np.abs(z) * np.tanh(1.5 * np.abs(z))).astype(np.complex64).ravel()
    H = 0.1
    a = (-0.5 * H * (np.arange(Ny) * 0.5 - 0.25 * (Ny - 1)))[:, None] + np.zeros((Ny, Nx - 1))
    b = (0.5 * H * (np.arange(Nx) * 0.5 - 0.25 * (Nx - 1)))[None, :] + np.zeros((Ny - 1, Nx))
    ab = np.concatenate([a.ravel(), b.ravel()]).astype(np.float32)
    ref, _, sw64 = run(Nx, Ny, np.float64, (psi.astype(complex), ab.astype(float), None, None), kappa, 64, 20)
    assert np.linalg.norm(ref) < 0.5 * np.linalg.norm(psi)
    err = []
    for wg in (0, 64):
        p, _, sw = run(Nx, Ny, np.float32, (psi, ab, None, None), kappa, wg, 20)
        assert wg or np.array_equal(sw[:, 0], sw64[:, 0])
        err.append(np.linalg.norm(p - ref) / np.linalg.norm(ref))
    assert err[0] <= 1.1 * err[1]


# solves that end before, at and after the turn (the sweep limit), and steps of
# few sweeps, which carry changes from the first one on
@pytest.mark.parametrize("dt,max_sweeps", [(0.1, 1), (0.1, 2), (0.1, 3), (0.1, 4), (0.1, 9), (1e-3, 1024), (4e-3, 1024),
                                           (1e-2, 1024)])
@pytest.mark.parametrize("kappa", [0.0, 5.0])
def test_fp32_short_solves(dt, max_sweeps, kappa):
    """Six steps stay within 5e-7 of 64 bits: each is rounded some ten times
    at 3e-8 of psi, in sums that the next steps do not amplify."""
    Nx, Ny = 150, 131
    f = state(Nx, Ny, np.float32, True, seed=9)
    f64 = (f[0].astype(complex), f[1].astype(float), f[2], f[3].astype(float))
    ref, ab64, sw64 = run(Nx, Ny, np.float64, f64, kappa, 8, 6, dt=dt, max_sweeps=max_sweeps)
    p, ab, sw = run(Nx, Ny, np.float32, f, kappa, 0, 6, dt=dt, max_sweeps=max_sweeps)
    assert np.array_equal(sw[:, 0], sw64[:, 0])
    assert np.linalg.norm(p - ref) <= 5e-7 * np.linalg.norm(ref)
    assert np.linalg.norm(ab - ab64) <= 5e-7 * np.linalg.norm(ab64)
