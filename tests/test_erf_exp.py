"""The occupations' erf and exponential (erf_table.h, physics.h): the table against
erf at 40 digits at every interval's edges, middle and in between, and on the
device the integrands whose arguments reach the table's ends and the
exponential's: widths sigma from a step to a slope over all masses, thresholds at
and beyond the mass range, slopes beta that over- and underflow.

Table: interpolation error below 1e-17 and eleven roundings of terms of at most
0.0625 x 1.13, 2^-53 of each: 1e-17 + 11 x 0.071 x 1.1e-16 < 1e-16.  Integrands: the
parity tests' bounds, and where an occupation is itself a rounding of 1 + erf (1e-16
of its full value), 1e-12 of the largest value."""
import os
import re

import numpy as np
import pytest

from conftest import ARCMIN, ROOT, T, say


def test_erf_table():
    mpmath = pytest.importorskip("mpmath")
    mpmath.mp.dps = 40
    src = open(os.path.join(ROOT, "g3lhalo_amd", "csrc", "erf_table.h")).read()
    rows = re.findall(r"\{(-?\d[^{}]*)\}", src)
    assert len(rows) == 48
    for i, row in enumerate(rows):
        c = [float(v) for v in row.split(",")]
        assert len(c) == 12
        for f in (0.0, 0.2, 0.5, 0.9, 1.0):
            x = (i + f) / 8
            t = x - (i + 0.5) / 8
            p = c[11]
            for v in c[10:1:-1]:
                p = p * t + v
            # the row's last addition is exact here: hi and the rest apart
            e = mpmath.mpf(p * t + c[0]) + mpmath.mpf(c[1]) - mpmath.erf(mpmath.mpf(x))
            assert abs(e) < 1e-16, (i, f, e)


@pytest.mark.gpu
@pytest.mark.parametrize("sigma,mth,beta", [(0.01, 1e13, 1.0), (0.4, 1e11, 0.0), (8.0, 1e13, 1.0),
                                            (0.1, 1e15, 1.0), (0.5, 1e12, 40.0),
                                            (0.5, 1e12, -40.0)])
def test_occupations(tables, sigma, mth, beta):
    import oracle as O
    from g3lhalo_amd import _lib
    hod = (0.5, 1.0, mth, sigma, 10 ** 13.3, beta)
    m = O.Model(tables)
    m.set_hods(hod, hod, A=0.3, eps=0.2, identical=False)
    ctx = _lib.Context(tables)
    sid = ctx.hodset(hod, hod, A=0.3, eps=0.2)
    rng = np.random.default_rng(int(1000 * sigma))
    b = m.borders()
    theta = np.array([1.0, 2.0, 4.0]) * ARCMIN
    for stat, term in ((0, 1), (0, 2), (1, 1), (1, 2), (1, 3)):
        lo = np.array([-1, -1, 0] + [np.log10(b[2])] * term + [b[0]])
        hi = np.array([6, 6, 6.28318] + [np.log10(b[3])] * term + [b[1]])
        x = lo + (hi - lo) * rng.random((4000, len(lo)))
        say(f"occupations sigma={sigma} mth={mth:g} beta={beta} stat={stat} term={term}")
        f = ctx.integrand(_lib.make_request(stat, term, theta, hodset=sid, type1=1, type2=2), x)
        f0 = m.integrand(stat, term, theta, x, 1, 2)
        assert np.array_equal(np.isfinite(f), np.isfinite(f0))
        ok = np.isfinite(f0)
        d = np.abs(f - f0)[ok] / (np.abs(f0[ok]) + 1e-12 * np.abs(f0[ok]).max() + 1e-300)
        print("max", d.max(), "p99.9", np.quantile(d, 0.999))
        assert np.quantile(d, 0.999) < 1e-10
        assert d.max() < 1e-5
    ctx.close()
