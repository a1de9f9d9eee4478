"""Coordinates and lattice vectors that are no finite numbers (a trajectory that has blown up) are
refused before anything is launched, and the next geometry is taken as usual."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("where", ["first", "last", "lattice"])
def test_not_finite_is_refused(bad, where):
    from dftbplus_amd import api, synth
    geo, params, opts = synth.workload("diamond1")
    x, lat = geo.coords.copy(), geo.latvecs.copy()
    if where == "lattice":
        lat[1, 1] = bad
    else:
        x[0 if where == "first" else -1, 2] = bad
    with pytest.raises(api.DftbHipError, match="finite"):
        api.neighbour_list(x, lat, 12.0)
    dp = api.DftbPlus(params, geo, opts)
    e = dp.get_energy()
    with pytest.raises(api.DftbHipError, match="finite"):
        dp.set_geometry(x, lat)
    dp.set_geometry(geo.coords, geo.latvecs)
    assert abs(dp.get_energy() - e) < 1e-10 * abs(e)
    dp.close()
