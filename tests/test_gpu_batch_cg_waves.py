"""The FP32-mixed batched CG gives instances of more than 4096 nodes sixteen
waves and the others four; FP64 four. In batches that mix them: FP64, the
first iteration of an instance among many is the oracle's steepest descent to
the line minimum; FP32-mixed, an instance among many ends at the FP64 form's
free energy, and in the bits it ends in alone."""
import numpy as np
import pytest

from tests.test_gpu_batch_cg import F, exact_jacobian_A, make, state

pytestmark = pytest.mark.gpu
nat = pytest.importorskip("svirl_amd._native")

from oracle import gl_oracle as O  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def _init():
    nat.init(0)


def batch(n, dtype, init):
    """An instance each at the ends of n - 2 small ones."""
    from svirl_amd import GLSolver
    filler = [GLSolver(Nx=4, Ny=5, dx=0.5, dy=0.5, order_parameter='random', random_seed=k, gl_parameter=5.0,
                       homogeneous_external_field=0.2, dtype=dtype) for k in range(n - 2)]
    return [make(0, 65, 40, 5.0, 0.3, dtype, init)] + filler + [make(1, 33, 29, 5.0, 0.1, dtype, init)]


# fewer and more instances than 256 CUs
@pytest.mark.parametrize("n", [3, 300])
def test_first_iteration_is_line_minimum(n):
    from svirl_amd.batch import BatchCG
    sims = batch(n, np.float64, 'random')
    ends = [sims[0], sims[-1]]
    before = [state(gl) for gl in ends]
    iters, _, _ = BatchCG(sims).cg(max_iter=1, rtol=0.0)
    assert np.all(iters == 1)
    for gl, (g, psi0, ab0, mt, em, k2, H) in zip(ends, before):
        _, psi1, ab1, *_ = state(gl)
        d = -O.jacobian_psi(g, k2, 0.0, em, H, mt, psi0, None, ab0)
        dA = -exact_jacobian_A(g, k2, H, mt, psi0, ab0)
        dp = psi1 - psi0
        ap = np.vdot(d, dp).real / np.vdot(d, d).real
        aA = np.dot(dA, ab1 - ab0) / np.dot(dA, dA)
        assert ap > 0 and aA > 0
        assert np.linalg.norm(dp - ap * d) <= 1e-10 * np.linalg.norm(ap * d)
        assert np.linalg.norm(ab1 - ab0 - aA * dA) <= 1e-10 * np.linalg.norm(aA * dA)
        f = lambda x, y: F(g, k2, em, H, mt, psi0 + x * d, ab0 + y * dA)
        fa = f(ap, aA)
        assert fa < f(0.0, 0.0)
        for sx in (0.9, 1.1):
            for sy in (0.9, 1.0, 1.1):
                assert fa <= f(sx * ap, sy * aA) + 1e-12 * abs(fa)


# 2600 and 957 nodes (four waves) beside 4355 (sixteen), and fewer or more
# instances than the 256 CUs hold at once
@pytest.mark.parametrize("n", [3, 300, 1100])
def test_fp32_mixed_reaches_fp64_energy(n):
    from svirl_amd.batch import BatchCG

    def sims(n, dtype):
        b = batch(n, dtype, 1.0)
        return b[:1] + [make(2, 65, 67, 5.0, 0.2, dtype, 1.0)] + b[1:]

    s64, s32 = sims(3, np.float64), sims(n, np.float32)
    alone = sims(3, np.float32)
    BatchCG(s64).cg(max_iter=3000, rtol=1e-6)
    iters, _, _ = BatchCG(s32).cg(max_iter=3000, rtol=1e-4)
    for k, a, b in ((0, s32[0], s64[0]), (1, s32[1], s64[1]), (-1, s32[-1], s64[-1])):
        fa, fb = a.observables.free_energy_fp64(), b.observables.free_energy_fp64()
        assert abs(fa - fb) <= 1e-5 * abs(fb)
        it1, _, _ = BatchCG([alone[k]]).cg(max_iter=3000, rtol=1e-4)
        assert it1[0] == iters[k]
        assert np.array_equal(alone[k].vars.order_parameter, a.vars.order_parameter)
