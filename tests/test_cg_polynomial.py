"""The line search's polynomial evaluation equals numpy's polyval2d to the
bit, in both working precisions, infinities and NaN included. CPU only."""
import numpy as np
import pytest

from numpy.polynomial.polynomial import polyder, polyval2d


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("scale", [1.0, 1e30, 1e-30])
def test_equals_polyval2d(dtype, scale):
    from svirl_amd.solvers.cg import polynomial_2d
    rng = np.random.default_rng(3)
    c = (scale * rng.normal(size=(5, 5))).astype(dtype)
    c[3, 1:] = c[4, 1:] = 0.0
    points = np.concatenate([rng.normal(size=(200, 2)) * 10.0 ** rng.integers(-8, 9, size=(200, 1)),
                             [[0.0, 0.0], [-0.0, 1.0], [np.inf, 0.5], [0.5, -np.inf], [np.nan, 1.0], [1e200, 1e200]]])
    with np.errstate(all="ignore"):
        for v in (c, polyder(c, axis=0), polyder(c, axis=1)):
            p = polynomial_2d(v)
            for alpha in points:
                want = np.float64(polyval2d(alpha[0], alpha[1], v))
                got = np.float64(p(float(alpha[0]), float(alpha[1])))
                assert want.tobytes() == got.tobytes() or (np.isnan(want) and np.isnan(got)), (alpha, want, got)
