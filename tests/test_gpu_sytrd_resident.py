"""The tridiagonalisation of matrices that fit on the chip, at the edges of its shapes: one
workgroup (up to 128 columns), workgroups exchanging vectors (up to 2560, with 256 or 512 threads
and 1 to 8 columns per thread), and the hand-over from the blocked form above that."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(n, kind):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    a = a + a.T
    if kind == "graded":      # rows over twelve orders of magnitude
        s = 10.0 ** np.linspace(-6, 6, n)
        a = a * s[:, None] * s[None, :]
    elif kind == "decoupled":  # columns whose part below the subdiagonal is zero: tau = 0
        a[np.abs(np.subtract.outer(np.arange(n), np.arange(n))) > 1] = 0.0
    elif kind == "tiny":       # sums of squares below the range of the fast reciprocal root
        a = a * 1e-150
    return np.asfortranarray(a)


def _similar(a, r, d, e, tau):
    """max |Q^T A Q - T| and max |Q^T Q - 1| for the stored reflectors."""
    n = len(d)
    q = np.eye(n)
    for c in range(n - 2, -1, -1):
        v = np.zeros(n)
        v[c + 1] = 1.0
        v[c + 2:] = r[c + 2:, c]
        q -= tau[c] * np.outer(v, v @ q)
    t = np.diag(d) + np.diag(e, 1) + np.diag(e, -1)
    return np.max(np.abs(q.T @ a @ q - t)), np.max(np.abs(q.T @ q - np.eye(n)))


# backward error of n Householder steps: a few n eps |A| (norm), growing slowly in practice
@pytest.mark.parametrize("kind", ["full", "graded", "decoupled", "tiny"])
@pytest.mark.parametrize("n", [2, 3, 31, 32, 33, 64, 65, 127, 128, 129, 130, 255, 256, 257, 513])
def test_resident_reduction_is_similarity(n, kind):
    from dftbplus_amd import api
    a = _matrix(n, kind)
    r, d, e, tau = api.dsytrd(a)
    scale = np.linalg.norm(a, 2)
    sim, orth = _similar(a, r, d, e, tau)
    eps = np.finfo(float).eps
    assert sim <= 4 * n * eps * scale
    assert orth <= 4 * n * eps
    assert np.array_equal(np.diag(r), d) and np.array_equal(np.diag(r, -1), e)


@pytest.mark.parametrize("n", [1024, 1025, 2048, 2049, 2560, 2561, 2700])
def test_resident_spectrum(n):
    from dftbplus_amd import api
    a = _matrix(n, "full")
    _, d, e, _ = api.dsytrd(a)
    import scipy.linalg
    w = scipy.linalg.eigvalsh_tridiagonal(d, e)
    ref = np.linalg.eigvalsh(a)
    assert np.max(np.abs(w - ref)) <= 4 * n * np.finfo(float).eps * np.max(np.abs(ref))


@pytest.mark.parametrize("n", [128, 700, 1500])
def test_resident_reduction_repeats_bit_for_bit(n):
    """Sums run in a fixed order: two runs of one matrix give the same bits."""
    from dftbplus_amd import api
    a = _matrix(n, "full")
    first, second = api.dsytrd(a), api.dsytrd(a)
    assert all(np.array_equal(x, y) for x, y in zip(first, second))
