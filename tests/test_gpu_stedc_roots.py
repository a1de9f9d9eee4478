"""Divide and conquer on spectra whose secular roots lie many orders of magnitude nearer to a pole
than the poles to each other: levels within 1e-6 of each other, and over twelve orders. The rational
iteration gives up on some of them and the bracket is halved, from the pole upwards."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("kind", ["close", "graded"])
@pytest.mark.parametrize("n", [37, 64, 100, 200])
def test_roots_next_to_a_pole(n, kind):
    from dftbplus_amd import api
    for seed in range(40):
        rng = np.random.default_rng([n, seed])
        if kind == "close":
            d, e = np.ones(n), 1e-6 * rng.standard_normal(n - 1)
        else:
            d = 10.0 ** -rng.uniform(0, 12, n)
            e = np.sqrt(d[1:] * d[:-1]) * rng.uniform(-1, 1, n - 1)
        w, z = api.dstedc(d, e)
        t = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
        # LAPACK dstedc's bound, a modest multiple of eps |T| per level of the tree
        tol = 160 * EPS * np.log2(n)
        assert np.max(np.abs(t @ z - z * w)) <= tol * np.max(np.abs(w)), seed
        assert np.max(np.abs(z.T @ z - np.eye(n))) <= tol, seed
