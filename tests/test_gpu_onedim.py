"""The one-kernel 1-D integrals (n_bar of an HOD set) against the reference's
adaptive quadrature written out here: the heap of src/hcubature.cpp:904-1021
over the GK15 rule of :695-757, every point value taken from the device
integrand (g3l_integrand, term 0), so that both refine the same function bit
for bit.

Bin counts: 2 (one jump), 17 and 128 (a few hundred regions), 300 and 400
(more than 1024 regions, more nodes than a block holds for its integrals), and
1000, where the jumps of the nearest-index mass function need more than the
2048 regions an integral may hold.

Both sides add the same at most 2048 region values, each a sum of 15 products:
they can differ by the order of those additions only, so by less than 4096
half-ulps of a sum of one sign, 5e-13 relative."""
import heapq
import math

import numpy as np
import pytest

from conftest import T, say

pytestmark = pytest.mark.gpu

XGK = (0.991455371120812639206854697526329, 0.949107912342758524526189684047851,
       0.864864423359769072789712788640926, 0.741531185599394439863864773280788,
       0.586087235467691130294144838258730, 0.405845151377397166906606412076961,
       0.207784955007898467600689403773245, 0.0)
WG = (0.129484966168869693270611432679082, 0.279705391489276667901467771423780,
      0.381830050505118944950369775488975, 0.417959183673469387755102040816327)
WGK = (0.022935322010529224963732008058970, 0.063092092629978553290700663189204,
       0.104790010322250183839876322541518, 0.140653259715525918745189590510238,
       0.169004726639267902826583426598550, 0.190350578064785409913256402421014,
       0.204432940075298892414161999234649, 0.209482141084727828012999174891714)


def _points(c, h):
    """Centre, then -/+ pairs of the seven-point rule's nodes, then the rest."""
    xs = [c]
    for j in (1, 3, 5, 0, 2, 4, 6):
        xs += [c - h * XGK[j], c + h * XGK[j]]
    return xs


def _rule(f, h):
    js = (1, 3, 5, 0, 2, 4, 6)
    rk, rg, rabs = f[0] * WGK[7], f[0] * WG[3], abs(f[0] * WGK[7])
    for n, j in enumerate(js):
        a, b = f[1 + 2 * n], f[2 + 2 * n]
        if n < 3:
            rg += WG[n] * (a + b)
        rk += WGK[j] * (a + b)
        rabs += WGK[j] * (abs(a) + abs(b))
    mean = 0.5 * rk
    rasc = WGK[7] * abs(f[0] - mean)
    for n, j in enumerate(js):
        rasc += WGK[j] * (abs(f[1 + 2 * n] - mean) + abs(f[2 + 2 * n] - mean))
    err, rabs, rasc = abs(rk - rg) * h, rabs * h, rasc * h
    if rasc != 0 and err != 0:
        scale = (200 * err / rasc) ** 1.5
        err = rasc * scale if scale < 1 else rasc
    if rabs > 2.2250738585072014e-308 / (50 * 2.220446049250313e-16):
        err = max(err, 50 * 2.220446049250313e-16 * rabs)
    return rk * h, err


def _adaptive(ctx, req, lo, hi, reltol, cap):
    """Value, or None when the integral needs more than cap regions."""
    def evaluate(regions):
        x = np.array([p for c, h in regions for p in _points(c, h)])[:, None]
        f = ctx.integrand(req, x).reshape(len(regions), 15)
        return [_rule(list(map(float, row)), h) for row, (c, h) in zip(f, regions)]
    c, h = 0.5 * (lo + hi), 0.5 * (hi - lo)
    (v, e), = evaluate([(c, h)])
    heap = [(-e, c, h, v)]
    while True:
        val = math.fsum(r[3] for r in heap)
        err = math.fsum(-r[0] for r in heap)
        thr = abs(val) * reltol
        if not (err > 0 and err > thr):
            return val
        new = []
        while heap:
            e0, c, h, v = heapq.heappop(heap)
            err = math.fsum(-r[0] for r in heap)
            new += [(c - 0.5 * h, 0.5 * h), (c + 0.5 * h, 0.5 * h)]
            if not (err > 0 and err > thr):
                break
        if len(heap) + len(new) > cap:
            return None
        for (c, h), (v, e) in zip(new, evaluate(new)):
            heapq.heappush(heap, (-e, c, h, v))


@pytest.mark.parametrize("nbins", [2, 17, 128, 300, 400, 1000])
def test_nbar_matches_adaptive_quadrature(nbins):
    from g3lhalo_amd import _lib
    say(f"onedim: nbins={nbins}")
    t = T.make_tables(nbins)
    hods = T.hod_prior_draws(2, seed=nbins)
    ctx = _lib.Context(t)
    lo = math.log10(t.mmin)
    hi = math.log10(math.exp(math.log(t.mmin) + math.log(t.mmax / t.mmin) * (nbins - 1) / nbins))
    if nbins >= 1000:
        with pytest.raises(_lib.G3LError) as e:
            ctx.hodset(hods[0], hods[1])
        assert _lib.STATUS_NAMES[e.value.rc] == "ENOMEM_POOL"
        ctx.close()
        return
    sid = ctx.hodset(hods[0], hods[1])
    _, n1, n2 = ctx.densities(sid)
    for zi in sorted({0, nbins // 2, nbins - 1}):
        z = t.zmin + zi * (t.zmax - t.zmin) / nbins
        for slot, got in ((1, n1[zi]), (2, n2[zi])):
            req = _lib.make_request(0, 0, (z, 0, 0), hodset=sid, type1=slot)
            want = _adaptive(ctx, req, lo, hi, 1e-4, 2048)
            assert got == pytest.approx(math.log(10.0) * want, rel=5e-13), (zi, slot)
    ctx.close()
