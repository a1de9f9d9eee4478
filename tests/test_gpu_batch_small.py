"""The batch's smallest molecules: up to 16 orbitals, swept in LDS (alone or beside molecules above the
direct classes) or solved directly beside larger ones, and the rounding floor of both Jacobi
kernels."""
import copy
import dataclasses

import numpy as np
import pytest

from test_gpu_batch import _chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [list(range(1, 17)), [16], [225, 16, 3], [17, 16], [40, 5]])
def test_small_class_edges(sizes):
    """Two iterations (the second starts from the first one's vectors) against the single-molecule
    path. Tolerances as for the direct solver: backward errors of n eps |H|, gaps of the chains."""
    from dftbplus_amd import api, synth
    _, params, opts = synth.workload("molecules1")
    o = dataclasses.replace(opts, max_scc_iter=2)
    rng = np.random.default_rng(6)
    mols = [_chain(n, rng) for n in sizes]
    b = api.MoleculeBatch(params, mols, o)
    e = b.scc()
    g = b.gradients()
    for m, geo in enumerate(mols):
        dp = api.DftbPlus(params, geo, o)
        es, qs, gs = dp.get_energy(), dp.get_gross_charges(), dp.get_gradients()
        dp.close()
        assert abs(es - e[m]) / geo.natom < 1e-10
        assert np.max(np.abs(qs - b.charges[m])) < 1e-9
        assert np.max(np.abs(gs - g[m])) < 1e-8
    b.close()


@pytest.mark.parametrize("n", [13, 226])
def test_level_at_zero_converges(n):
    """A molecule of a Jacobi class with an eigenvalue at 0 Ha in its last iteration (all on-site
    energies shifted by what a secant search on the oracle finds): a pair touching a diagonal entry
    near 0 must not rotate on rounding noise until the sweep limit, which would be an error."""
    from dftbplus_amd import api, synth
    from oracle import dftb_ref as R
    _, params, opts = synth.workload("molecules1")
    o = dataclasses.replace(opts, max_scc_iter=3)
    geo = _chain(n, np.random.default_rng(7))

    def shifted(c):
        p = copy.deepcopy(params)
        for sp in p.species:
            sp.onsite = [x + c for x in sp.onsite]
        return p

    def level(c, k=None):
        e = R.Calculator(shifted(c), geo, o).scc().eigenvalues
        k = int(np.argmin(np.abs(e))) if k is None else k
        return e[k], k

    f0, k = level(0.0)
    c0, c1 = 0.0, -f0
    for _ in range(8):
        f1, _ = level(c1, k)
        if abs(f1) < 1e-12:
            break
        c0, c1, f0 = c1, c1 - f1 * (c1 - c0) / (f1 - f0), f1
    assert abs(f1) < 1e-10
    p = shifted(c1)
    b = api.MoleculeBatch(p, [geo], o)
    e = b.scc()
    res = R.Calculator(p, geo, o).scc()
    assert abs(res.energy_mermin - e[0]) / geo.natom < 1e-8
    assert np.max(np.abs(res.charges - b.charges[0])) < 1e-8
    b.close()
