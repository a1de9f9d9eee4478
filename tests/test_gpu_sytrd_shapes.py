"""The shapes of the register-resident tridiagonalisation that several problems of one size select
(many rows per workgroup, 256 or 512 threads), and its FP32 form, at sizes that leave remainders."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REAL = np.array([[a, b, c] for a in (0, 0.5) for b in (0, 0.5) for c in (0, 0.5)])


def _crystal(norb):
    """Carbons, and one to three hydrogens for the remainder, on a jittered cubic lattice."""
    from dftbplus_amd import synth
    from dftbplus_amd.model import Geometry
    _, params, opts = synth.workload("diamond1")
    spec = np.array([0] * (norb // 4) + [1] * (norb % 4))
    side = int(np.ceil(len(spec) ** (1 / 3)))
    rng = np.random.default_rng(norb)
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[: len(spec)]
    x = 3.4 * g + rng.uniform(-0.2, 0.2, (len(spec), 3))
    return Geometry(x, spec[rng.permutation(len(spec))], np.eye(3) * 3.4 * side), params, opts


# rows of a problem (twice the orbitals at complex points), problems, and the shape for 256 compute
# units: threads, rows and columns per workgroup
@pytest.mark.parametrize("norb, points, shape", [
    (250, 8, (256, 8, 1)), (125, -12, (256, 16, 1)), (123, -24, (256, 32, 1)),
    (401, 8, (256, 16, 2)), (201, -12, (256, 32, 2)), (601, 3, (256, 8, 4)),
    (601, 4, (256, 16, 4)), (602, 8, (512, 32, 2)), (1021, 8, (512, 32, 2)),
    (1101, 2, (512, 16, 4)), (1101, 3, (512, 16, 4)),
])
def test_problems_side_by_side(norb, points, shape):
    """Together against one by one, after one iteration: levels to backward errors of n eps |H|
    (1e-12), charges to what kT = 0.01 Ha makes of them."""
    from dftbplus_amd import api
    geo, params, opts = _crystal(norb)
    if points > 0:
        k = REAL[:points]
    else:
        k = np.random.default_rng(1).uniform(0.05, 0.45, (-points, 3))
    o = dataclasses.replace(opts, kpoints=k, max_scc_iter=1)
    out = []
    try:
        for mode in (1, 0):
            api.set_tuning(2, mode)
            dp = api.DftbPlus(params, geo, o)
            e, q = dp.get_energy(), dp.get_gross_charges()
            out.append((e / geo.natom, q, np.array([dp.get_eigenvalues_k(p)[0] for p in range(len(k))])))
            dp.close()
    finally:
        api.set_tuning(2, 1)
    for x, y, tol in zip(*out, (1e-10, 1e-9, 1e-11)):
        assert np.max(np.abs(x - y)) < tol, shape


@pytest.mark.parametrize("norb", [65, 130, 257, 301, 601, 1101, 2101])
def test_fp32_levels(norb):
    """FP32 iterations against FP64: the products of the reduction and the stored columns are rounded
    to FP32, the sums of the tridiagonalisation are FP64. A level moves by the mean of those
    independent roundings over its vector, eps32 |H|; 16 times that for the condition of S and the
    worst of all levels."""
    from dftbplus_amd import api
    geo, params, opts = _crystal(norb)
    o = dataclasses.replace(opts, max_scc_iter=1)
    out = []
    for kw in (dict(), dict(precision=1, refine_below=0.0)):
        dp = api.DftbPlus(params, geo, o, **kw)
        dp.get_energy()
        out.append(dp.get_eigenvalues()[0])
        dp.close()
    d = np.max(np.abs(out[0] - out[1]))
    assert 0 < d <= 16 * np.finfo(np.float32).eps * np.max(np.abs(out[0]))
