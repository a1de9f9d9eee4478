"""k-points solved together against one by one, with real and complex points in one mesh: two
groups of different size, below and above one block of 128 reflectors."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [1, 2])
def test_mixed_mesh_together_equals_one_by_one(cells):
    """32 and 256 orbitals, 64 and 512 in the complex points' embedding. Both solve the same
    problems to n eps |H| (1e-13); one iteration hands that on to charges and forces."""
    from dftbplus_amd import api, synth
    geo, params, opts = synth.workload(f"diamond{cells}")
    k = np.array([[0, 0, 0], [0.5, 0, 0.5], [0.25, 0, 0], [0.125, 0.25, 0.375], [0.5, 0.25, 0]])
    opts = dataclasses.replace(opts, kpoints=k, max_scc_iter=2)
    out = []
    try:
        for mode in (1, 0):
            api.set_tuning(2, mode)
            dp = api.DftbPlus(params, geo, opts)
            out.append((dp.get_energy(), dp.get_gross_charges(), dp.get_gradients(),
                        np.concatenate([dp.get_eigenvalues_k(q)[0] for q in range(len(k))])))
            dp.close()
    finally:
        api.set_tuning(2, 1)
    for x, y in zip(*out):
        assert np.max(np.abs(np.asarray(x) - np.asarray(y))) < 1e-10
