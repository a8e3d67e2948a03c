"""The row-marching solves of a single grid (an explicit workgroup count) on
grids that run on register tiles by default: a large grid against the oracle,
and a timed-out run."""
import numpy as np
import pytest

from tests.test_gpu_solver import gl_ab, gl_psi, oracle_of, rel

pytestmark = pytest.mark.gpu
nat = pytest.importorskip("svirl_amd._native")


@pytest.fixture(scope="module", autouse=True)
def _init():
    nat.init(0)


def test_large_grid_rows_match_oracle():
    """Long row ranges per wave, fused passes and a team of several dozen
    workgroups; sweep counts exact, fields within 1e-10 of the oracle."""
    from svirl_amd import GLSolver, workloads
    gl = GLSolver(Nx=769, Ny=641, dx=0.5, dy=0.5, order_parameter='random', random_seed=3, gl_parameter=5.0,
                  normal_conductivity=200.0, homogeneous_external_field=0.05, dtype=np.float64)
    c = gl.cfg
    gl.mesh.material_tiling = workloads.holes_mask(int(c.Nxc), int(c.Nyc), 0.5, 0.5, seed=5)
    gl.vars.set_order_parameter_to_zero_outside_material()
    gl.params.linear_coefficient = workloads.pinning_field(int(c.Nx), int(c.Ny), 0.5, seed=6)
    st = oracle_of(gl)
    gl.solve._init_td()
    td = gl.solve._td
    td.wg = td._default_wg()
    assert td.wg > 16
    gl.solve.td(dt=0.05, Nt=3)
    st.td(dt=0.05, Nt=3)
    assert td.sweeps == st.sweeps
    assert rel(gl_psi(gl), st.psi) < 1e-10 and rel(gl_ab(gl), st.ab) < 1e-10


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_rows_barrier_timeout_reports_and_keeps_state(dtype):
    from svirl_amd import GLSolver
    gl = GLSolver(Nx=300, Ny=200, dx=0.5, dy=0.5, order_parameter='random', random_seed=5, gl_parameter=2.0,
                  normal_conductivity=10.0, homogeneous_external_field=0.1, dtype=dtype)
    gl.solve._init_td()
    gl.solve._td.wg = 8
    psi0 = np.array(gl.vars.order_parameter, copy=True)
    st = oracle_of(gl)
    nat.call("glx_td_force_barrier_abort")
    with pytest.raises(nat.GLXError) as err:
        gl.solve.td(dt=0.1, Nt=3)
    assert err.value.code == nat.GLX_E_TIMEOUT and "timed out" in str(err.value)
    assert gl.solve._td.sweeps == []
    assert np.array_equal(gl.vars.order_parameter, psi0)
    gl.solve.td(dt=0.1, Nt=3)
    st.td(dt=0.1, Nt=3)
    tol = 1e-10 if dtype == np.float64 else 1e-4
    if dtype == np.float64:
        assert gl.solve._td.sweeps == st.sweeps
    assert rel(gl_psi(gl), st.psi) < tol and rel(gl_ab(gl), st.ab) < tol
