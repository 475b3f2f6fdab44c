"""Timed cases of the NNMap / NMapMap path: what a user's program calls.

A case is one call pattern of the reference's drivers and fit loop, at the
sizes of this repository's configurations, tests and benchmark, through the
public entry points of the C ABI (``g3lhalo_amd._lib``).  ``listed()`` gives
the fixed cases, ``draw(rng)`` more of the same ranges; ``prepare`` makes what
the program holds before the call (tables in HBM, HOD sets, requests),
``run`` is one pass and returns its outputs, ``work`` the bytes and flops a
pass cannot do without, and ``exact`` the values that have a closed or
one-dimensional form, in plain numpy.

Call patterns ("call"):

``plain``      one term after another (``NNMap_Model::NNMap``,
               ``NMapMap_Model::NMapMap``): host-driven integrals.
``batch``      a list of integrals at once (``calculateNNMap.x``,
               ``calculateNMapMap.x``, a configuration's sweep).
``fit``        one step of a fit (``NNMap_Model::calculateAll``): a new HOD
               pair, its densities, then every term at the three type pairs.
``nbar``       n_bar(z) of new HOD sets alone.
``precompute`` the input tables from a cosmology (``doPrecomputations.x``).
``serve``      requests that arrive while others refine (the server).
"""
from __future__ import annotations

import functools
import math
import random

import numpy as np
import torch

from g3lhalo_amd import _lib, flops
from g3lhalo_amd import tables as T

TYPE_PAIRS = ((1, 2), (1, 1), (2, 2))
# the drivers' tolerances per term (NNMap 1h, 2h, 3h; NMapMap) and the
# configurations' common one
DRIVER_TOL = {0: (1e-3, 1e-3, 1e-4), 1: (1e-3, 1e-3, 1e-3)}
CONFIG_TOL = (1e-4, 1e-4, 1e-4)
MAXEVAL = 5000000


def _case(call, **kw):
    c = {"call": call, "nbins": 128}
    c.update(kw)
    return c


def listed():
    return [
        # NNMap_Model::NNMap of one aperture triplet: three integrals, one
        # after another, as a script that asks for single values has it
        dict(_case("plain", stat=0, triplets=1, driver_tol=True, maxeval=MAXEVAL),
             name="plain_triplet"),
        # the drivers' small example: a thetas file of four triplets, all
        # three terms at the drivers' tolerances
        dict(_case("batch", stat=0, triplets=4, driver_tol=True, maxeval=MAXEVAL, mixed=False),
             name="driver_4"),
        # calculateAll for one triplet and for eleven (an equal-aperture data
        # vector): a new red/blue HOD pair with a correlated NsatNsat term
        dict(_case("fit", triplets=1, maxeval=MAXEVAL), name="fit_step_1"),
        dict(_case("fit", triplets=11, maxeval=MAXEVAL), name="fit_step_11"),
        # the fit sweep's data vector for one HOD vector
        dict(_case("batch", stat=0, triplets=55, driver_tol=False, maxeval=MAXEVAL, mixed=False),
             name="nnmap_55"),
        # the headline workload: 550 triplets, 1e-4
        dict(_case("batch", stat=0, triplets=550, driver_tol=False, maxeval=MAXEVAL, mixed=False),
             name="nnmap_550"),
        # the galaxy-shear-shear statistic, a ragged part of its 550 triplets
        dict(_case("batch", stat=1, triplets=137, driver_tol=False, maxeval=MAXEVAL,
                   mixed=False), name="nmapmap_137"),
        # the 256-bin tables in the mixed-precision form
        dict(_case("batch", stat=0, triplets=55, driver_tol=False, maxeval=MAXEVAL, mixed=True,
                   nbins=256), name="mixed_256bin_55"),
        # a new HOD set: what every fit step pays first
        dict(_case("nbar", sets=1), name="nbar_1"),
        # the HOD sweep's 256 sets in one call
        dict(_case("nbar", sets=256), name="nbar_256"),
        # doPrecomputations.x on the model's 128-bin grid
        dict(_case("precompute"), name="precompute_128"),
        # the served stream: eight requests, each submitted while the earlier
        # ones refine
        dict(_case("serve", requests=8, triplets=12, maxeval=MAXEVAL), name="serve_8"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    call = rng.choice(("plain", "batch", "batch", "batch", "fit", "nbar", "precompute", "serve"))
    nbins = rng.choice((64, 100, 128, 256))
    if call == "plain":
        return _case(call, nbins=nbins, stat=rng.randrange(2), triplets=rng.randint(1, 5),
                     driver_tol=rng.random() < 0.5, maxeval=_log_int(rng, 2e5, MAXEVAL))
    if call == "batch":
        return _case(call, nbins=nbins, stat=rng.randrange(2), triplets=_log_int(rng, 1, 500),
                     driver_tol=rng.random() < 0.5, maxeval=_log_int(rng, 2e5, MAXEVAL),
                     mixed=rng.random() < 0.25)
    if call == "fit":
        return _case(call, nbins=nbins, triplets=_log_int(rng, 1, 55),
                     maxeval=_log_int(rng, 2e5, MAXEVAL))
    if call == "nbar":
        return _case(call, nbins=nbins, sets=_log_int(rng, 1, 256))
    if call == "precompute":
        return _case(call, nbins=rng.randint(16, 128))
    return _case(call, nbins=nbins, requests=rng.randint(2, 8), triplets=_log_int(rng, 1, 30),
                 maxeval=_log_int(rng, 2e5, MAXEVAL))


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=None)
def _tables(nbins):
    return T.make_tables(nbins)


def _rng(case, seed):
    return np.random.default_rng([seed & 0x7fffffff, 7])


def _thetas(rng, n):
    """n aperture triplets [rad], log-uniform over the configurations' range."""
    return 0.5 * 64.0 ** rng.uniform(0.0, 1.0, (n, 3)) * T.ARCMIN_IN_RAD


def _hods(rng, n):
    return T.hod_prior_draws(n, seed=int(rng.integers(1 << 31)))


def _tols(case):
    return DRIVER_TOL[case.get("stat", 0)] if case.get("driver_tol", True) else CONFIG_TOL


def _cosmology(case, seed):
    """A cosmology near the fiducial one, the model's grids and a source n(z)."""
    rng = _rng(case, seed)
    om = rng.uniform(0.25, 0.35)
    cosmo = {"Omega_m": om, "Omega_Lambda": 1.0 - om, "Omega_b": rng.uniform(0.04, 0.05),
             "sigma8": rng.uniform(0.7, 0.9), "H0": rng.uniform(65.0, 75.0),
             "ns": rng.uniform(0.94, 0.98)}
    z = np.linspace(0.01, 3.0, 100)
    nz = z ** 2 * np.exp(-(z / rng.uniform(0.4, 0.6)) ** 1.5)
    nz /= nz.sum() * (z[-1] - z[0]) / len(z)
    return cosmo, (0.001, 2.0, 1e10, 1e17, 1e-4, 1e4), z, nz


def _serve_requests(case, seed):
    """Requests in turn: NNMap at one type pair, NMapMap, both statistics'
    2-halo terms, and a two-population request at the three type pairs."""
    rng = _rng(case, seed)
    out = []
    for i in range(case["requests"]):
        h = _hods(rng, 2)
        two = i % 4 == 3
        terms = (((0, 1), (0, 2), (0, 3)), ((1, 1), (1, 2), (1, 3)), ((0, 2), (1, 2)),
                 ((0, 1), (0, 2), (0, 3)))[i % 4]
        ints = [(st, t, th, p) for th in _thetas(rng, case["triplets"]) for st, t in terms
                for p in (TYPE_PAIRS if two else ((1, 2),))]
        out.append((h[0], h[1] if two else h[0], two, ints))
    return out


def prepare(case, seed):
    call = case["call"]
    if call == "precompute":
        cosmo, grid, z, nz = _cosmology(case, seed)
        return {"case": case, "args": (cosmo, *grid, case["nbins"], z, nz)}
    s = {"case": case, "ctx": _lib.Context(_tables(case["nbins"]))}
    ctx = s["ctx"]
    if call == "serve":
        s["reqs"] = _serve_requests(case, seed)
        s["srv"] = _lib.Server(ctx)
        return s
    rng = _rng(case, seed)
    if call == "nbar":
        s["hods"] = (_hods(rng, case["sets"]), _hods(rng, case["sets"]))
        return s
    h = _hods(rng, 2)
    if call == "fit":
        # the pair of the step and its NsatNsat correlation; requests refer to
        # the one set that the step makes (id 0 after the clear)
        s["hod"] = (h[0], h[1], float(rng.uniform(0.0, 0.3)), float(rng.uniform(0.0, 0.2)))
        sid, pairs, stat = 0, TYPE_PAIRS, 0
    else:
        sid, pairs, stat = ctx.hodset(h[0], h[1]), ((1, 2),), case["stat"]
    tol = _tols(case)
    s["reqs"] = [_lib.make_request(stat, t, th, hodset=sid, type1=p[0], type2=p[1],
                                   reltol=tol[t - 1], maxeval=case["maxeval"])
                 for p in pairs for th in _thetas(rng, case["triplets"]) for t in (1, 2, 3)]
    return s


# -------------------------------------------------------------------- pass
def _results(res):
    return {"value": np.array([r.value for r in res]), "raw": np.array([r.raw for r in res]),
            "err": np.array([r.err for r in res]),
            "neval": np.array([r.neval for r in res], dtype=np.int64),
            "rounds": np.array([r.rounds for r in res], dtype=np.int64),
            "status": np.array([r.status for r in res], dtype=np.int64)}


def _clear(ctx):
    _lib.check("g3l_hodset_clear", _lib.load().g3l_hodset_clear(ctx.h))


def run(state):
    case = state["case"]
    call = case["call"]
    if call == "precompute":
        return _lib.precompute(*state["args"])
    ctx = state["ctx"]
    if call == "plain":
        return _results([ctx.eval_plain(r) for r in state["reqs"]])
    if call == "batch":
        return _results(ctx.eval_batch(state["reqs"],
                                       precision=_lib.MIXED if case["mixed"] else _lib.FP64))
    if call == "fit":
        _clear(ctx)
        h1, h2, a, eps = state["hod"]
        sid = ctx.hodset(h1, h2, A=a, eps=eps)
        rho, n1, n2 = ctx.densities(sid)
        out = _results(ctx.eval_batch(state["reqs"]))
        out.update(rho_bar=rho, n_bar1=n1, n_bar2=n2)
        return out
    if call == "nbar":
        _clear(ctx)
        first = ctx.hodsets(*state["hods"])
        d = [ctx.densities(first + i) for i in range(case["sets"])]
        return {"rho_bar": np.stack([x[0] for x in d]), "n_bar1": np.stack([x[1] for x in d]),
                "n_bar2": np.stack([x[2] for x in d])}
    # serve: each request's HOD set is made when it arrives, two rounds after
    # the one before
    _clear(ctx)
    srv = state["srv"]
    done = {}
    for tag, (h1, h2, two, ints) in enumerate(state["reqs"]):
        sid = ctx.hodset(h1, h2, identical=not two)
        srv.submit([_lib.make_request(st, t, th, hodset=sid, type1=p[0], type2=p[1], reltol=1e-4,
                                      maxeval=case["maxeval"]) for st, t, th, p in ints], tag)
        for _ in range(2):
            srv.step()
            done.update(srv.poll())
    while len(done) < len(state["reqs"]):
        srv.step()
        done.update(srv.poll())
    return _results([r for tag in sorted(done) for r in done[tag]])


# -------------------------------------------------------------------- work
# GK15 evaluations of one n_bar(z) and of one precomputation integral, on
# average, and flops of a precomputation evaluation by the convention of
# g3lhalo_amd.flops (window, transfer function, P(k)).
NBAR_EVALS, PRECOMP_EVALS, PRECOMP_FLOPS = 400, 400, 300


def _table_bytes(nbins):
    return 8 * (6 * nbins + 4 * nbins * nbins + nbins)


def work(case):
    call, nb = case["call"], case["nbins"]
    if call == "precompute":
        n = 1 + nb + 100 + 2 * nb * nb + 256 * nb
        return {"bytes": 8 * (200 + 6 * nb + 4 * nb * nb),
                "flops": n * PRECOMP_EVALS * PRECOMP_FLOPS}
    nbar = 2 * nb * NBAR_EVALS * flops.FLOPS_PER_EVAL[0]
    if call == "nbar":
        return {"bytes": 8 * nb * nb + 24 * nb * case["sets"], "flops": case["sets"] * nbar}
    if call == "serve":
        ints = [(st, t) for _, _, _, x in _serve_requests(case, 0) for st, t, _, _ in x]
        extra = case["requests"] * nbar
    else:
        stat = case.get("stat", 0)
        pairs = 3 if call == "fit" else 1
        ints = [(stat, t) for _ in range(pairs * case["triplets"]) for t in (1, 2, 3)]
        extra = nbar if call == "fit" else 0
    # the integrals stop at the evaluation cap
    return {"bytes": _table_bytes(nb) + len(ints) * 112,
            "flops": extra + sum(case["maxeval"] * flops.flops_per_eval(st, t)
                                 for st, t in ints)}


# ------------------------------------------------------------ exact values
def _nbar_exact(case, hods):
    """n_bar(z_i) = ln 10 int m n(m, z_i) (Ncen + Nsat) dlog10 m over the mass
    range of the model, n(m, z) by nearest index: piecewise constant between
    the mass bins' midpoints, so each piece is a smooth integral."""
    t, nb = _tables(case["nbins"]), case["nbins"]
    lnr = math.log(t.mmax / t.mmin)
    # borders of the pieces in units of bins: 0, 1/2, 3/2, ..., nb - 1
    edge = np.concatenate([[0.0], np.arange(nb - 1) + 0.5, [nb - 1.0]])
    x, wx = np.polynomial.legendre.leggauss(24)
    mid, half = 0.5 * (edge[1:] + edge[:-1]), 0.5 * (edge[1:] - edge[:-1])
    lm = math.log(t.mmin) + (mid[:, None] + half[:, None] * x) * lnr / nb   # ln m
    m = np.exp(lm)
    hmf = t.hmf.reshape(nb, nb)
    out = np.empty((len(hods), nb))
    for i, (_, alpha, mth, sigma, mprime, beta) in enumerate(hods):
        e = 1 + torch.erf(torch.from_numpy((lm - math.log(mth)) / sigma / 1.414213562)).numpy()
        occ = 0.5 * alpha * e + 0.5 * e * (m / mprime) ** beta
        piece = (m * occ * wx).sum(axis=1) * half * lnr / nb   # d ln m = ln 10 dlog10 m
        out[i] = hmf @ piece
    return out


def _rho_exact(case):
    """Omega_m(z) rho_crit on the redshift grid."""
    t = _tables(case["nbins"])
    c = t.cosmo
    a = (1 + t.zmin + np.arange(t.nbins) * (t.zmax - t.zmin) / t.nbins) ** 3
    return c.Omega_m * a / (c.Omega_m * a + c.Omega_Lambda) * c.rho_crit


def _precompute_exact(case, seed):
    """Grids, distances and lensing efficiency; the other tables have no form
    short of the adaptive integrals themselves."""
    cosmo, (zmin, zmax, mmin, mmax, kmin, kmax), nz_z, nz_n = _cosmology(case, seed)
    n, c_kms = case["nbins"], 299792.0
    i = np.arange(n)
    z = zmin + i * (zmax - zmin) / n

    def hubble_distance(x):
        return c_kms / cosmo["H0"] / np.sqrt(cosmo["Omega_m"] * (1 + x) ** 3
                                             + cosmo["Omega_Lambda"])
    x, wx = np.polynomial.legendre.leggauss(40)

    def distance(zz):
        return 0.5 * zz * (hubble_distance(0.5 * np.outer(zz, 1 + x)) * wx).sum(axis=1)
    w, ws = distance(z), distance(nz_z)
    dz = (nz_z[-1] - nz_z[0]) / len(nz_z)
    g = np.where(nz_z >= z[:, None], nz_n * (ws - w[:, None]) / ws, 0.0).sum(axis=1) * dz
    return {"z": z, "m": mmin * np.exp(i * math.log(mmax / mmin) / n),
            "k": kmin * np.exp(i * math.log(kmax / kmin) / n), "w": w, "dwdz": hubble_distance(z),
            "g": g, "hmf": None, "P_lin": None, "b_h": None, "concentration": None}


def exact(case, seed):
    call = case["call"]
    if call == "precompute":
        return _precompute_exact(case, seed)
    rng = _rng(case, seed)
    if call == "nbar":
        a, b = _hods(rng, case["sets"]), _hods(rng, case["sets"])
        return {"rho_bar": np.tile(_rho_exact(case), (case["sets"], 1)),
                "n_bar1": _nbar_exact(case, a), "n_bar2": _nbar_exact(case, b)}
    if call == "fit":
        h = _hods(rng, 2)
        none = dict.fromkeys(("value", "raw", "err", "neval", "rounds", "status"))
        return {**none, "rho_bar": _rho_exact(case), "n_bar1": _nbar_exact(case, h[:1])[0],
                "n_bar2": _nbar_exact(case, h[1:])[0]}
    # the 5- to 7-dimensional integrals are defined by their refinement: no
    # value but the reference algorithm's own
    return None
