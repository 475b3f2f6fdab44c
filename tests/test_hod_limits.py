"""HOD parameters and arguments at the ends of their ranges.  A quotient by a known
reciprocal (one product and one residual) is NaN where an operand is infinite; the
occupations, densities and look-ups have to be there what divisions give:

* sigma infinite: a flat occupation, erf(0);
* M_th infinite: an empty population, no galaxies and a density of zero;
* a mass that underflows to zero or overflows, an infinite redshift (g3l_integrand):
  the outermost table entry on that side."""
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, T, say


def test_host_expressions(tmp_path):
    exe = str(tmp_path / "limits_probe")
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-x", "hip",
                        "--offload-arch=gfx950", "-Wno-unused-command-line-argument",
                        os.path.join(ROOT, "tests", "cxx", "limits_probe.cpp"), "-o", exe],
                       capture_output=True, text=True)
    if r.returncode:
        pytest.skip("hipcc host build unavailable: " + r.stderr[-300:])
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    assert int(out.split()[-2]) > 600
    assert int(out.split()[-1]) == 0, out


def _hod(**kw):
    p = dict(zip(("f", "alpha", "mth", "sigma", "mprime", "beta"), T.FIDUCIAL_HOD), **kw)
    return tuple(p[k] for k in ("f", "alpha", "mth", "sigma", "mprime", "beta"))


@pytest.mark.gpu
def test_infinite_sigma(tables):
    """Twice the integrals' tolerance of 1e-4 from the oracle's densities, and finite
    terms."""
    import oracle as O
    from g3lhalo_amd import _lib
    h = _hod(sigma=float("inf"))
    ctx = _lib.Context(tables)
    say("limits: sigma infinite")
    sid = ctx.hodset(h, T.FIDUCIAL_HOD)
    m = O.Model(tables)
    m.set_hods(h, T.FIDUCIAL_HOD)
    for got, want in zip(ctx.densities(sid), m.densities()):
        np.testing.assert_allclose(got, want, rtol=2e-4)
    for prec in (_lib.FP64, _lib.MIXED):
        res = ctx.eval_batch([_lib.make_request(0, t, (1e-3, 1e-3, 2e-3), hodset=sid, maxeval=2000)
                              for t in (1, 2, 3)], precision=prec)
        assert all(np.isfinite(r.value) for r in res)
    ctx.close()


@pytest.mark.gpu
def test_infinite_threshold(tables):
    from g3lhalo_amd import _lib
    ctx = _lib.Context(tables)
    say("limits: M_th infinite")
    a = ctx.densities(ctx.hodset(_hod(mth=float("inf")), T.FIDUCIAL_HOD))
    b = ctx.densities(ctx.hodset(T.FIDUCIAL_HOD, T.FIDUCIAL_HOD))
    assert not a[1].any()
    np.testing.assert_array_equal(a[2], b[2])
    ctx.close()


@pytest.mark.gpu
def test_arguments_beyond_the_tables():
    """n_bar's integrand at masses and redshifts of no table entry, with a mass function
    that has no zeros (an infinite mass times one would be NaN)."""
    from g3lhalo_amd import _lib
    t = T.make_tables()
    t.hmf = np.maximum(t.hmf, 1e-30)
    ctx = _lib.Context(t)
    sid = ctx.hodset(T.FIDUCIAL_HOD, T.FIDUCIAL_HOD)
    say("limits: integrand beyond the tables")

    def f(z, x):
        return ctx.integrand(_lib.make_request(0, 0, (z, 0, 0), hodset=sid, type1=1),
                             np.array(x)[:, None])
    inf = float("inf")
    np.testing.assert_array_equal(f(0.3, [-inf, -400.0]), [0.0, 0.0])
    assert np.all(np.isposinf(f(0.3, [inf, 400.0])))
    x = [11.0, 13.3, 15.0]
    np.testing.assert_array_equal(f(inf, x), f(100.0, x))
    np.testing.assert_array_equal(f(-inf, x), f(-100.0, x))
    assert np.any(f(inf, x) != f(-inf, x))
    ctx.close()
