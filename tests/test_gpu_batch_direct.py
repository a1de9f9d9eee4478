"""The molecule batch's direct eigensolver (up to 224 orbitals) and its hand-over to Jacobi sweeps
above, against the single-molecule path after one and two SCC iterations (the second one reuses
the factor of the overlap and skips what has converged)."""
import dataclasses

import numpy as np
import pytest

from test_gpu_batch import _chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,iters", [
    ([1], 1),                                   # no column to reduce, no merge
    ([1, 2, 3, 16, 17, 31, 32, 33, 64, 65], 2),   # leaves of the divide and conquer; small shapes
    ([128, 129, 224, 225, 240], 2),             # largest shapes, Jacobi above
    ([9] * 70 + [64], 2),                       # more molecules than one launch's compute units
])
def test_direct_eigensolver_edges(sizes, iters):
    """Tolerances: both paths solve the same pencil with backward errors of n eps |H| (1e-13 Ha
    at 240 orbitals); gaps of the chains amplify it by less than 1e3 in the charges."""
    from dftbplus_amd import api, synth
    _, params, opts = synth.workload("molecules1")
    o = dataclasses.replace(opts, max_scc_iter=iters)
    rng = np.random.default_rng(5)
    mols = [_chain(n, rng) for n in sizes]
    b = api.MoleculeBatch(params, mols, o)
    e = b.scc()
    g = b.gradients()
    for m in sorted({sizes.index(n) for n in sizes} | {len(sizes) - 1}):
        dp = api.DftbPlus(params, mols[m], o)
        es, qs, gs = dp.get_energy(), dp.get_gross_charges(), dp.get_gradients()
        dp.close()
        assert abs(es - e[m]) / mols[m].natom < 1e-10
        assert np.max(np.abs(qs - b.charges[m])) < 1e-9
        assert np.max(np.abs(gs - g[m])) < 1e-8
    b.close()
