"""Register tiles on grids with dx != dy, a size for every tile shape, single
and batched, against the row-marching solves (an explicit workgroup count):
FP64 to the bit. FP32 to 5e-6 after three steps: the rounding of a few dozen
sweeps (2e-7 in the mean, six times that at the worst of 1e6 nodes) and a stop
rule of 1e-6 that the rows' rounded differences may meet a sweep apart (what is
left of the solve there, 1e-6 / (1 - 0.6))."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
nat = pytest.importorskip("svirl_amd._native")

SIZES = [(33, 29), (130, 111), (300, 257), (410, 602), (1000, 900)]


@pytest.fixture(scope="module", autouse=True)
def _init():
    nat.init(0)


def solver(size, k, dtype):
    from svirl_amd import GLSolver
    Nx, Ny = size
    rng = np.random.default_rng(50 + k)
    gl = GLSolver(Nx=Nx, Ny=Ny, dx=0.5, dy=0.4, order_parameter='random', random_seed=k + 1,
                  gl_parameter=np.inf if k % 3 == 2 else 4.0, normal_conductivity=200.0,
                  homogeneous_external_field=0.02, dtype=dtype)
    if k % 2:
        gl.mesh.material_tiling = rng.random((Nx - 1, Ny - 1)) > 0.05
        gl.vars.set_order_parameter_to_zero_outside_material()
        gl.params.linear_coefficient = 1.0 + 0.2 * rng.normal(size=(Nx, Ny))
    return gl


def by_rows(size, k, dtype):
    gl = solver(size, k, dtype)
    gl.solve._init_td()
    gl.solve._td.wg = 32
    gl.solve.td(dt=0.1, Nt=3)
    return gl


def compare(gl, g1, dtype):
    p, p1 = gl.vars.order_parameter, g1.vars.order_parameter
    pairs = [(p.real, p1.real), (p.imag, p1.imag)] + list(zip(gl.vars.vector_potential, g1.vars.vector_potential))
    if dtype == np.float64:
        assert gl.solve._td.sweeps == g1.solve._td.sweeps
        assert all(np.array_equal(x, y) for x, y in pairs)
    else:
        assert np.all(np.isfinite(p1))
        assert max(np.max(np.abs(x - y)) for x, y in pairs) <= 5e-6


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_unequal_spacings(dtype):
    from svirl_amd.batch import BatchTD
    rows = [by_rows(s, k, dtype) for k, s in enumerate(SIZES)]
    single = [solver(s, k, dtype) for k, s in enumerate(SIZES)]
    batch = [solver(s, k, dtype) for k, s in enumerate(SIZES)]
    b = BatchTD(batch)
    assert not any(b.on_teams())
    b.td(dt=0.1, Nt=3)
    for gl, gb, g1 in zip(single, batch, rows):
        gl.solve.td(dt=0.1, Nt=3)
        compare(gl, g1, dtype)
        compare(gb, g1, dtype)
