"""The device neighbour list beyond the sizes of its short forms: more neighbours than are ranked
by counting (1024), and more candidate images than one pass of the scans' tiles (2^21)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_rank_and_bitonic_orders_equal_oracle():
    """365 to 2974 neighbours per atom: both sorts in one call, bit for bit."""
    from dftbplus_amd import api, synth
    from oracle import dftb_ref as R
    geo, _, _ = synth.workload("diamond1")
    ref = R.neighbour_list(geo.coords, geo.latvecs, 30.0)
    call, i2c, neigh, d2 = api.neighbour_list(geo.coords, geo.latvecs, 30.0)
    assert max(len(v) for v in neigh) > 2048 > 1024 > min(len(v) for v in neigh)
    assert np.array_equal(call, ref.coords_all) and np.array_equal(i2c, ref.img2cent)
    for a in range(len(neigh)):
        assert np.array_equal(neigh[a], ref.neigh[a])
        assert np.array_equal(d2[a], ref.dist2[a])


def test_many_candidate_images():
    """9000 atoms in a flat cell, 2.5 million candidates, against a k-d tree over the images that
    can lie within the cutoff (distances to rounding: 1e-9, coordinates of 1000 bohr at 1e-13 times 2 x 20)."""
    from dftbplus_amd import api
    from scipy.spatial import cKDTree
    rng = np.random.default_rng(3)
    lat = np.diag([900.0, 900.0, 5.0])
    cut = 20.0
    x = rng.uniform(size=(9000, 3)) @ lat
    call, i2c, neigh, d2 = api.neighbour_list(x, lat, cut)
    tr = np.array([[a, b, c] for a in (0, -1, 1) for b in (0, -1, 1)
                   for c in (0, -5, -4, -3, -2, -1, 1, 2, 3, 4, 5)]) @ lat
    pts = (tr[:, None, :] + x[None]).reshape(-1, 3)
    near = cKDTree(pts).query_ball_point(x, cut)
    for a in range(len(x)):
        idx = np.array(near[a])
        idx = idx[(idx % len(x) >= a) & (idx != a)]
        want = np.sort(np.sum((pts[idx] - x[a]) ** 2, axis=1))
        assert len(d2[a]) == 1 + len(want) and neigh[a][0] == a
        assert np.allclose(d2[a][1:], want, rtol=0, atol=1e-9)
        assert np.allclose(np.sum((call[neigh[a]] - x[a]) ** 2, axis=1), d2[a], rtol=0, atol=1e-9)
        assert np.all(i2c[neigh[a]] >= a)
