"""Divide and conquer is as good relative to the matrix whatever its units: one leaf, the first
merges and several heights, from the edge of the denormal numbers to that of the range."""
import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("scale", [1e-300, 1e-150, 1e-100, 1e-9, 1e-3, 1.0, 1e3, 1e99, 1e160, 1e300])
@pytest.mark.parametrize("n", [1, 16, 17, 40, 64, 65, 200, 700])
def test_any_units(n, scale):
    from dftbplus_amd import api
    rng = np.random.default_rng(n)
    d, e = rng.standard_normal(n), rng.standard_normal(max(n - 1, 0))
    w, z = api.dstedc(d * scale, e * scale)
    w = w / scale
    t = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
    ref = scipy.linalg.eigvalsh_tridiagonal(d, e) if n > 1 else d
    # LAPACK dstedc's bounds, a modest multiple of eps |T| per level of the tree; the reference's own
    # scaling by a number that is no power of two is one rounding more
    tol = 160 * EPS * max(1.0, np.log2(max(n, 2))) * np.max(np.abs(ref))
    assert np.max(np.abs(w - ref)) <= tol
    assert np.max(np.abs(t @ z - z * w)) <= tol
    assert np.max(np.abs(z.T @ z - np.eye(n))) <= tol
