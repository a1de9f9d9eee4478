"""The Slater-Koster interpolation to the last bit: its roundings are part of the result, because
past the end of a table a second difference over 1e-5 is divided by 1e-10, which makes 1e-11 of an
ulp. The reference does each rounding as the kernel writes it out, with exactly rounded fma's."""
import math
from fractions import Fraction

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DELTA = 1.0e-5


def _fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def _interval(i0, dx, xx):
    x0 = i0 * dx
    return min(max(math.ceil(_fma(-float(i0), dx, xx) * (1.0 / _fma(float(i0 + 1), dx, -x0))), 1), 8)


def _neville(col, i0, dx, xx, icl):
    x = [_fma(float(i0 + i), dx, -xx) for i in range(8)]
    cc = [float(col[i0 - 1 + i]) for i in range(8)]
    dd = list(cc)
    x0 = i0 * dx
    delta = [1.0 / (_fma(float(i0 + i + 1), dx, -x0) if i < 2 else (i0 + i + 1) * dx - x0)
             for i in range(7)]
    yy, icl, r2 = cc[icl - 1], icl - 1, [0.0] * 8
    for mm in range(1, 8):
        for ii in range(8 - mm):
            diff = _fma(r2[ii], x[ii + 1], -cc[ii + 1]) if mm == 2 else dd[ii] - cc[ii + 1]
            r2[ii] = diff * delta[mm - 1]
            cc[ii], dd[ii] = x[ii] * r2[ii], x[ii + mm] * r2[ii]
        if 2 * icl < 8 - mm:
            yy += cc[icl]
        else:
            icl -= 1
            yy += dd[icl]
    return yy


def _integral(col, dx, r):
    """Value and the bound of its error: 0 in the table, past it a few roundings of the terms."""
    n = len(col)
    if r >= _fma(float(n), dx, 1.0):
        return 0.0, 0.0
    ind = math.floor(r / dx)
    if ind < n:
        i0 = max(min(n, ind + 4), 8) - 7
        return _neville(col, i0, dx, r, _interval(i0, dx, r)), 0.0
    y = []
    for x in (_fma(float(n), dx, -DELTA), _fma(float(n), dx, DELTA)):
        y.append(_neville(col, n - 7, dx, x, _interval(n - 7, dx, x)))
    y1 = float(col[n - 1])
    p, pp = (y[1] - y[0]) / (2.0 * DELTA), (y[1] + y[0] - 2.0 * y1) / (DELTA * DELTA)
    a3, a4, a5 = 10 * y1 + 4 * p + 0.5 * pp, -15 * y1 - 7 * p - pp, 6 * y1 + 3 * p + 0.5 * pp
    t = -(r - _fma(float(n), dx, 1.0))
    scale = 15 * abs(y1) + 7 * abs(p) + abs(pp)
    return ((a5 * t + a4) * t + a3) * t * t * t, 16 * np.finfo(float).eps * scale


def test_s_blocks_to_the_last_bit():
    """All pairs of s atoms on a line (the distance is then exact), from the first rows of the table,
    where the interpolation is off its middle interval, over its end to the cutoff."""
    from conftest import reference_arrays
    from dftbplus_amd import api, synth
    from dftbplus_amd.model import Geometry
    from oracle import dftb_ref as R
    _, params, opts = synth.workload("molecules1")
    h = next(k for k, s in enumerate(params.species) if list(s.shells) == [0])
    dx, rows = params.dist, params.ham[(h, h)].shape[0]
    end = rows * dx
    x = np.cumsum([0.0, 1.7, 0.061, 2 * dx + 0.013, 1.9, 0.83, 2.31, 1.17, end - 8.0, 0.0301, 0.25, 0.21])
    coords = np.zeros((len(x), 3))
    coords[:, 0] = x
    calc = R.Calculator(params, Geometry(coords, np.full(len(x), h), None), opts)
    H, S = api.build_h0_s(api.SkHandle(params), reference_arrays(calc))
    seen = [0, 0, 0]
    for k in range(len(calc.sp.at1)):
        a, b = calc.sp.at1[k], calc.sp.img2[k]
        if a == b:
            continue
        r = abs(x[b] - x[a])
        seen[0 if r < 4 * dx else 1 if r < end else 2] += 1
        for out, tab in ((H, params.ham[(h, h)]), (S, params.over[(h, h)])):
            v, bound = _integral(tab[:, 0], dx, r)
            assert abs(out[calc.sp.start[k]] - v) <= bound, (r, out[calc.sp.start[k]], v)
    assert min(seen) > 0, seen
