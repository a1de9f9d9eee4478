"""Slater-Koster blocks and pair forces of dimers over the whole range of the tables, both
derivative modes: the first rows (interpolation off its middle interval), grid points, the last
rows, the tail to zero and beyond it, for s-s, s-p and p-p pairs in both orders."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
def test_dimers_equal_oracle(mode):
    """Energies and forces of one SCC iteration to 1e-9: the formulas are the oracle's, the step of
    the difference quotients is 1e-4 bohr (1e-16 / 1e-4 in a derivative; mode 1 has no quotients, and
    theirs are off by h^2 times a third derivative over 6, up to 1e-7 at short distances)."""
    from dftbplus_amd import api, synth
    from dftbplus_amd.model import Geometry
    from oracle import dftb_ref as R
    _, params, opts = synth.workload("molecules1")
    o = dataclasses.replace(opts, max_scc_iter=1)
    end = params.ham[(0, 0)].shape[0] * params.dist
    rng = np.random.default_rng(4)
    mols = []
    for pair in ((0, 0), (0, 1), (1, 0), (1, 2)):
        for r in (1.7, 100 * params.dist, 3.0031, end - 4.5 * params.dist, end - 2.5 * params.dist,
                  end - 0.5 * params.dist, end + 0.3, end + 0.99, end + 1.5):
            u = rng.normal(size=3)
            mols.append(Geometry(np.array([np.zeros(3), r * u / np.linalg.norm(u)]),
                                 np.array(pair, dtype=np.int64), None))
    b = api.MoleculeBatch(params, mols, o, force_mode=mode)
    e, g = b.scc(), b.gradients()
    b.close()
    for m, geo in enumerate(mols):
        c = R.Calculator(params, geo, o)
        res = c.scc()
        assert abs(res.energy_mermin - e[m]) < 1e-9, (m, geo.coords)
        assert np.max(np.abs(c.gradients(res) - g[m])) < (1e-9 if mode == 0 else 1e-7), m
