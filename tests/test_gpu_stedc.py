"""Divide and conquer at the edges of its tree (leaves of up to 16 rows, heights 0 to 7) and on spectra
that deflate nothing, much or everything."""
import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _tridiagonal(n, kind):
    rng = np.random.default_rng(n)
    d, e = rng.standard_normal(n), rng.standard_normal(max(n - 1, 0))
    if kind == "wilkinson":          # glued: pairs of levels equal to rounding
        d = np.abs(np.arange(n) % 21 - 10.0)
        e = np.ones(max(n - 1, 0))
        e[20::21] = 1e-9
    elif kind == "toeplitz":         # no deflation
        d, e = 2.0 * np.ones(n), -np.ones(max(n - 1, 0))
    elif kind == "graded":
        g = 10.0 ** np.linspace(0, -12, n)
        d, e = d * g, e * np.sqrt(g[:-1] * g[1:])
    elif kind == "constant":         # a multiple of the identity: everything deflates
        d, e = 3.0 * np.ones(n), np.zeros(max(n - 1, 0))
    elif kind == "split":            # zero couplings at and off the tears
        e[::7] = 0.0
        if n > 2:
            e[n // 2 - 1] = 0.0
    return d, e


@pytest.mark.parametrize("kind", ["random", "wilkinson", "toeplitz", "graded", "constant", "split"])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 66, 127, 129, 257, 700, 1030])
def test_divide_and_conquer(n, kind):
    from dftbplus_amd import api
    d, e = _tridiagonal(n, kind)
    w, z = api.dstedc(d, e)
    t = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
    ref = scipy.linalg.eigvalsh_tridiagonal(d, e) if n > 1 else d
    scale = np.max(np.abs(ref))
    # LAPACK dstedc's bounds: a modest multiple of eps |T| per tree level
    tol = 40 * EPS * max(1.0, np.log2(max(n, 2)))
    assert np.all(np.diff(w) >= 0)
    assert np.max(np.abs(w - ref)) <= tol * scale
    assert np.max(np.abs(t @ z - z * w)) <= 4 * tol * scale
    assert np.max(np.abs(z.T @ z - np.eye(n))) <= 4 * tol


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("n", [20, 200])
def test_values_that_are_no_numbers_are_an_error(n, bad):
    from dftbplus_amd import api
    d, e = _tridiagonal(n, "random")
    d[n // 3] = bad
    with pytest.raises(api.DftbHipError):
        api.dstedc(d, e)
    w, _ = api.dstedc(*_tridiagonal(n, "random"))   # and the next call is unaffected
    assert np.all(np.isfinite(w))
