"""Batched TD on teams of workgroups (wg_per_cu > 0, and instances that no
register tile holds): graph replay, every pass depth, both precisions, a
timed-out run, and the autotuner, which times shapes only where instances run
on teams."""
import numpy as np
import pytest

from tests.test_gpu_batch import CASES, make, oracle_run

pytestmark = pytest.mark.gpu
nat = pytest.importorskip("svirl_amd._native")


@pytest.fixture(scope="module", autouse=True)
def _init():
    nat.init(0)


def fields(gl):
    a, b = gl.vars.vector_potential
    return np.array(gl.vars.order_parameter), np.array(a), np.array(b)


def big(dtype, kappa=5.0, seed=3):
    """One grid above what the registers hold."""
    from svirl_amd import GLSolver
    return GLSolver(Nx=1300, Ny=1210, dx=0.5, dy=0.5, order_parameter='random', random_seed=seed, gl_parameter=kappa,
                    normal_conductivity=200.0, homogeneous_external_field=0.01, dtype=dtype)


def test_explicit_workgroups_put_a_batch_on_teams():
    from svirl_amd.batch import BatchTD
    b = BatchTD([make(k, *c) for k, c in enumerate(CASES)])
    assert not any(b.on_teams()) and all(b.on_teams(1)) and all(b.on_teams(4))
    assert BatchTD([make(0, *CASES[0]), big(np.float64)]).on_teams() == [False, True]
    assert BatchTD([big(np.float32)]).on_teams() == [True]


@pytest.mark.parametrize("depth", [2, 3, 4])
@pytest.mark.parametrize("use_graph", [False, True])
def test_teams_match_oracle(depth, use_graph):
    from svirl_amd.batch import BatchTD
    sims = [make(k, *c) for k, c in enumerate(CASES)]
    refs = [oracle_run(gl, 0.1, 6) for gl in sims]
    b = BatchTD(sims, use_graph=use_graph)
    b.shape = (4 if use_graph else 1, 4, depth)
    b.td(dt=0.1, Nt=6)
    for gl, st in zip(sims, refs):
        assert [tuple(x) for x in gl.solve._td.sweeps] == st.sweeps
        assert np.max(np.abs(gl.flatten_array(gl.vars.order_parameter) - st.psi)) <= 1e-11
        if gl.params.solveA:
            a, b_ = gl.vars.vector_potential
            ab = np.concatenate([gl.flatten_a_array(a), gl.flatten_b_array(b_)])
            assert np.max(np.abs(ab - st.ab)) <= 1e-11


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("depth", [2, 3, 4])
def test_teams_fp32_close_to_single_rows(depth, noalloc):
    from svirl_amd.batch import BatchTD
    sims = [make(k, *c, dtype=np.float32) for k, c in enumerate(CASES)]
    alone = [make(k, *c, dtype=np.float32) for k, c in enumerate(CASES)]
    b = BatchTD(sims, noalloc=noalloc)
    b.shape = (2, 4, depth)
    b.td(dt=0.1, Nt=5)
    for gl, g1 in zip(sims, alone):
        g1.solve._init_td()
        g1.solve._td.wg = 4
        g1.solve.td(dt=0.1, Nt=5)
        assert np.all(np.abs(np.array(gl.solve._td.sweeps) - np.array(g1.solve._td.sweeps)) <= 1)
        assert np.max(np.abs(gl.vars.order_parameter - g1.vars.order_parameter)) <= 1e-5


def test_teams_barrier_timeout_keeps_states():
    """The aborted call makes one step, which writes only buffers that were
    not current."""
    from svirl_amd.batch import BatchTD
    sims = [make(k, *c) for k, c in enumerate(CASES)]
    before = [fields(gl) for gl in sims]
    refs = [oracle_run(gl, 0.1, 4) for gl in sims]
    b = BatchTD(sims, use_graph=False)
    b.shape = (2, 4, 3)
    nat.call("glx_td_force_barrier_abort")
    with pytest.raises(nat.GLXError) as err:
        b.td(dt=0.1, Nt=1)
    assert err.value.code == nat.GLX_E_TIMEOUT
    for gl, v0 in zip(sims, before):
        assert all(np.array_equal(x, y) for x, y in zip(fields(gl), v0))
    b.td(dt=0.1, Nt=4)
    for gl, st in zip(sims, refs):
        assert [tuple(x) for x in gl.solve._td.sweeps] == st.sweeps
        assert np.max(np.abs(gl.flatten_array(gl.vars.order_parameter) - st.psi)) <= 1e-11


def test_autotuner_leaves_batches_in_registers_alone():
    from svirl_amd.batch import BatchTD
    sims = [make(k, *c) for k, c in enumerate(CASES[:3])]
    b = BatchTD(sims, tune_steps=1)
    n = b.tune_need() + 1
    b.td(dt=0.1, Nt=n)
    assert b.timings == {}
    assert all(len(gl.solve._td.sweeps) == n for gl in sims)


def test_autotuner_times_shapes_of_teams():
    """One instance on teams beside one in registers; the fields are those of
    each alone."""
    from svirl_amd.batch import BatchTD
    sims, alone = ([make(1, *CASES[1]), big(np.float64, np.inf)] for _ in range(2))
    b = BatchTD(sims, tune_steps=1)
    n = b.tune_need() + 1
    b.td(dt=0.1, Nt=n)
    assert {k[2] for k in b.timings} == {2, 3, 4} and b.shape in b.timings
    for gl, g1 in zip(sims, alone):
        g1.solve.td(dt=0.1, Nt=n)
        assert gl.solve._td.sweeps == g1.solve._td.sweeps
        assert all(np.array_equal(x, y) for x, y in zip(fields(gl), fields(g1)))
