"""GEMM outputs at the sizes where another workgroup tile is chosen, and the triangular inverses
of the Cholesky and compact-WY kernels, through the entry points that use them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


# sizes around multiples of 32, 64 and 128 and of the tile choice (256 compute units)
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (31, 33, 17), (32, 32, 16), (65, 64, 5), (129, 127, 40),
                                   (573, 286, 573), (511, 1025, 64), (1030, 1031, 33), (2049, 130, 20)])
def test_gemm_tiles(m, n, k, ta, tb):
    from dftbplus_amd import api
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k) if ta == "N" else (k, m))
    b = rng.standard_normal((k, n) if tb == "N" else (n, k))
    c0 = rng.standard_normal((m, n))
    oa, ob = (a if ta == "N" else a.T), (b if tb == "N" else b.T)
    bound = (k + 2) * EPS * (np.abs(oa) @ np.abs(ob) + np.abs(c0))
    c = api.dgemm(a, b, ta, tb, 1.5, -0.5, c0)
    assert np.all(np.abs(c - (1.5 * oa @ ob - 0.5 * c0)) <= 2 * bound)


# Cholesky blocks of 64 with remainders; the reflectors of the back-transformation in blocks of
# 256 and halves of 128
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 129, 130, 200, 257, 258, 385, 513])
def test_sygvd_block_edges(n):
    import scipy.linalg
    from dftbplus_amd import api
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, n))
    s = x @ x.T / n + np.eye(n)
    h = rng.standard_normal((n, n))
    h = h + h.T
    w, c, l = api.sygvd(h, s)
    ref = scipy.linalg.eigh(h, s, eigvals_only=True)
    scale = max(1.0, np.abs(ref).max())
    tol = 40 * max(n, 8) * EPS       # condition of s is about 5
    assert np.max(np.abs(w - ref)) <= tol * scale
    assert np.max(np.abs(c.T @ s @ c - np.eye(n))) <= tol
    assert np.max(np.abs(h @ c - s @ c * w)) <= 4 * tol * scale * np.abs(s).max()
    lo = np.tril(l)
    assert np.max(np.abs(lo @ lo.T - s)) <= 4 * n * EPS * np.abs(s).max()


@pytest.mark.parametrize("n,bad", [(40, 0), (64, 63), (70, 64), (200, 137)])
def test_cholesky_reports_the_failing_minor(n, bad):
    from dftbplus_amd import api
    s = np.eye(n)
    s[bad, bad] = -1.0
    with pytest.raises(api.DftbHipError, match=f"info={n + bad + 1}"):
        api.sygvd(np.eye(n), s)


def test_padded_host_matrices():
    """Host arrays whose leading dimension exceeds n (the copies go column by column)."""
    import ctypes as C
    from dftbplus_amd import api
    n, ld = 70, 83
    rng = np.random.default_rng(1)
    h = rng.standard_normal((n, n))
    h = h + h.T
    a = np.zeros((ld, n), order="F")
    b = np.zeros((ld, n), order="F")
    a[:n], b[:n] = h, np.eye(n)
    w = np.zeros(n)
    api._check(api.lib().dftbhip_sygvd(1, b"V", b"L", n, api._d(a), ld, api._d(b), ld, api._d(w)), "sygvd")
    w0, c0, _ = api.sygvd(h, np.eye(n))
    assert np.array_equal(w, w0) and np.array_equal(a[:n], c0) and not a[n:].any()
