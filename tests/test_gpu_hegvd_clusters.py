"""The complex drop-in on large clusters of equal levels, where the last independent vectors of a
cluster keep little of their norm: Hermitian matrices of low rank, and with levels over ten orders."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("n", [40, 130, 300])
def test_low_rank(n):
    from dftbplus_amd import api
    for seed in range(4):
        rng = np.random.default_rng([n, seed])
        v = rng.standard_normal((n, n // 8)) + 1j * rng.standard_normal((n, n // 8))
        h = v @ v.conj().T
        x = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
        s = x @ x.conj().T / n + np.eye(n)
        w, c, _ = api.hegvd(np.asfortranarray(h), np.asfortranarray(s))
        scale = np.max(np.abs(w))
        # |S^-1| = 1: backward errors of n eps |H| and n eps |S|, and what the Gram-Schmidt of
        # vectors of remaining norm 1 / sqrt(m) keeps of them
        tol = 40 * n ** 1.5 * EPS
        assert np.max(np.abs(w[: n - n // 8])) <= tol * scale
        assert np.max(np.abs(h @ c - (s @ c) * w)) <= tol * scale * np.linalg.norm(s, 2)
        assert np.max(np.abs(c.conj().T @ s @ c - np.eye(n))) <= tol


def test_levels_over_ten_orders():
    """Clusters end where neighbours are 1e-8 apart, so vectors beside one are orthogonal to eps over
    that: 1e-5 allows for clusters that many levels chain together. Vectors keep the order of their
    levels, so the residuals stay at those of the solve."""
    from dftbplus_amd import api
    n = 520
    rng = np.random.default_rng([n, 1])
    a = rng.standard_normal((n, n))
    a = a + 1j * rng.standard_normal((n, n))
    g = 10.0 ** np.linspace(0, -10, n)
    h = g[:, None] * (0.5 * (a + a.conj().T)) * g[None, :]
    w, c, _ = api.hegvd(np.asfortranarray(h), np.asfortranarray(np.eye(n) + 0j))
    assert np.max(np.abs(c.conj().T @ c - np.eye(n))) <= 1e-5
    assert np.max(np.abs(h @ c - c * w)) <= 1e-7 * np.max(np.abs(w))
