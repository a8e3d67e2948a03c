"""Register tiles where the diagonal of a node outside the material vanishes:
dt eps = 1 makes 1 + dt (|psi|^2 - eps) zero at psi = 0, on the tiles' nodes
beyond the grid and in holes. The sweeps give 0 there, as the row-marching
solves (an explicit workgroup count) do: FP64 to the bit, FP32 to the
rounding of a few steps' sweeps (an ulp of 6e-8, 4 / (4 + |psi|^2) kept from
sweep to sweep) and a stop rule of 1e-6. (FP32 counts are not compared: the
solves take 200 to 450 sweeps, where 1e-7 of rounding moves a stop by some.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
nat = pytest.importorskip("svirl_amd._native")


@pytest.fixture(scope="module", autouse=True)
def _init():
    nat.init(0)


def solver(Nx, Ny, dtype, kappa, eps, seed):
    from svirl_amd import GLSolver
    gl = GLSolver(Nx=Nx, Ny=Ny, dx=1.0, dy=1.0, order_parameter='random', random_seed=seed, gl_parameter=kappa,
                  normal_conductivity=200.0, homogeneous_external_field=0.05, dtype=dtype)
    mt = np.ones((Nx - 1, Ny - 1), dtype=bool)
    mt[Nx // 3:Nx // 3 + 4, Ny // 2:Ny // 2 + 3] = False
    gl.mesh.material_tiling = mt
    gl.vars.set_order_parameter_to_zero_outside_material()
    if eps == 'map':  # 1 in the hole and along the grid's edges alone
        e = np.full((Nx, Ny), 0.9)
        e[Nx // 3 + 1:Nx // 3 + 4, Ny // 2 + 1:Ny // 2 + 3] = 1.0
        e[[0, -1], :] = 1.0
        e[:, [0, -1]] = 1.0
        gl.params.linear_coefficient = e
    return gl


def compare(gl, g1, dtype):
    assert np.all(np.isfinite(g1.vars.order_parameter))
    s, s1 = np.array(gl.solve._td.sweeps), np.array(g1.solve._td.sweeps)
    p, p1 = gl.vars.order_parameter, g1.vars.order_parameter
    if dtype == np.float64:
        assert np.array_equal(s, s1)
        assert np.array_equal(p, p1)
        assert all(np.array_equal(x, y) for x, y in zip(gl.vars.vector_potential, g1.vars.vector_potential))
    else:
        assert np.all(np.isfinite(p))
        assert np.max(np.abs(p - p1)) <= 2e-5


ALL = [(17, 12, np.inf, 1.0), (130, 70, 5.0, 1.0), (64, 40, 5.0, 'map'), (57, 100, np.inf, 'map')]


@pytest.mark.parametrize("case", range(len(ALL)))
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_tiles_equal_rows_at_zero_diagonal(case, dtype):
    Nx, Ny, kappa, eps = ALL[case]
    gl, g1 = (solver(Nx, Ny, dtype, kappa, eps, seed=case + 1) for _ in range(2))
    gl.solve.td(dt=1.0, Nt=3)
    g1.solve._init_td()
    g1.solve._td.wg = 8
    g1.solve.td(dt=1.0, Nt=3)
    compare(gl, g1, dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_batched_tiles_equal_rows_at_zero_diagonal(dtype):
    from svirl_amd.batch import BatchTD
    sims = [solver(*c[:2], dtype, c[2], c[3], seed=k + 1) for k, c in enumerate(ALL)]
    BatchTD(sims).td(dt=1.0, Nt=3)
    for k, (c, gl) in enumerate(zip(ALL, sims)):
        g1 = solver(*c[:2], dtype, c[2], c[3], seed=k + 1)
        g1.solve._init_td()
        g1.solve._td.wg = 8
        g1.solve.td(dt=1.0, Nt=3)
        compare(gl, g1, dtype)
