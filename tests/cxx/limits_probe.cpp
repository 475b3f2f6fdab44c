// Host build of the HOD occupations, the mass chain, the redshift factors and the F
// kernel (physics.h) at the ends of their parameters' ranges, against the same expressions
// with IEEE divisions: prints the number of values compared and every one that
// differs.
#include "../../g3lhalo_amd/csrc/physics.h"

#include <cmath>
#include <cstdio>

using namespace g3l;

static int count = 0, bad = 0;
static void same(const char *what, double got, double want) {
  ++count;
  if (got == want || (got != got && want != want)) return;
  ++bad;
  printf("%s: %g instead of %g\n", what, got, want);
}

int main() {
  const double inf = INFINITY;
  const double mmin = 1e10;
  for (double sigma : {1e-300, 0.3, 1e300, 1.7e308, inf})
    for (double mth : {1e-300, 1e12, 1e300, inf})
      for (double m : {0., 1e10, 3e13, 1e17, inf}) {
        DevHod h{1., 0.7, mth, sigma, 2e13, 1.1};
        Mass M{};
        M.m = m;
        M.L = std::log(m / mmin);
        const double rs = 1. / sigma, lth = std::log(mmin / mth), lmp = std::log(mmin / h.mprime);
        const double e = 1 + erf((M.L + lth) / sigma / 1.414213562);
        const double er = 1 + erf(std::log(m / mth) / sigma / 1.414213562);
        const Occ o = P64::occ(h, rs, lth, lmp, M), x = PMix::occ(h, rs, lth, lmp, M),
                  r = P64R::occ(h, rs, lth, lmp, M);
        same("P64 Ncen", o.nc, 0.5 * h.alpha * e);
        same("P64 Nsat", o.ns, 0.5 * e * std::exp(h.beta * (M.L + lmp)));
        same("PMix Ncen", x.nc, 0.5 * h.alpha * e);
        same("PMix Nsat", x.ns, 0.5 * e * std::exp(h.beta * (M.L + lmp)));
        same("P64R Ncen", r.nc, 0.5 * h.alpha * er);
        same("P64R Nsat", r.ns, 0.5 * er * std::pow(m / h.mprime, h.beta));
      }
  DevTables T{};
  T.nb = 128;
  T.mmin = mmin;
  T.mmax = 1e17;
  T.lmr = std::log(T.mmax / T.mmin);
  T.rmmin = 1. / T.mmin;
  T.rlmr = 1. / T.lmr;
  for (double x : {-inf, -400., 10., 13.7, 400., inf}) {
    double m, L;
    const double ix = mass_chain(T, x, m, L), want = std::pow(10., x);
    same("m", m, want);
    same("L", L, std::log(want / T.mmin));
    same("index", ix, std::log(want / T.mmin) * T.nb / T.lmr);
  }
  // zero and denormal densities: 1 / n_bar is infinite
  for (double n : {0., 1e-310, 1e-3})
    for (double rho : {8e10, inf}) {
      const double nb[1] = {n}, one[1] = {1.}, rh[1] = {rho}, rrho[1] = {1. / rho};
      T.rho = rh;
      T.rrho = rrho;
      T.dwdz = T.g = T.p1 = T.p2 = one;
      TermArgs a{};
      a.nb1 = nb;
      a.nb2 = one;
      double zpre, zfac;
      zfactors<kNN1>(T, a, 0, 0.3, 1., zpre, zfac);
      same("NNMap density factor", zpre, 1. / n / 1. / rho);
      zfactors<kNM1>(T, a, 0, 0.3, 1., zpre, zfac);
      same("NMapMap density factor", zpre, 1. / n / rho / rho);
    }
  // the bispectrum's kernel, whose k2 / k2 is one for either sign
  for (double k : {-inf, -1e300, -0.3, -1e-310, -0., 0., 1e-310, 0.3, 1e300, inf, (double)NAN})
    same("F", fkern(0.2, k, 0.5), 0.7143 + 0.2857 * 0.5 * 0.5 + 0.5 * 0.5 * (0.2 / k + k / k));
  printf("%d %d\n", count, bad);
}
