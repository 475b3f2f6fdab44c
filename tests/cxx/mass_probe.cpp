// Host build of mass_direct (physics.h) against mass_chain, and of kix_round against
// its chain with the library's logarithm: reads nb, log10 mmin, log10 mmax and a
// seed; prints the arguments taken directly, those of them whose indices differ from
// the chain's, the largest difference of the index argument, the largest relative
// error of the mass, the non-masses taken directly, and the k whose index differs.
#include "../../g3lhalo_amd/csrc/physics.h"

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

using namespace g3l;

int main(int argc, char **argv) {
  if (argc != 5) return 1;
  DevTables T{};
  T.nb = atoi(argv[1]);
  const double lo = atof(argv[2]), hi = atof(argv[3]);
  T.mmin = std::pow(10., lo);
  T.mmax = std::pow(10., hi);
  T.lmr = std::log(T.mmax / T.mmin);
  T.rmmin = 1. / T.mmin;
  T.rlmr = 1. / T.lmr;
  const long double lmm = std::log((long double)T.mmin);
  const double consts[DevTables::kConsts] = {(double)lmm, (double)(lmm - (double)lmm)};
  T.rrho = consts - T.nb;
  std::mt19937_64 rng(atoi(argv[4]));
  std::uniform_real_distribution<double> U(0, 1);
  long taken = 0, wrong = 0;
  double far = 0, err = 0;
  for (int i = 0; i < 400000; ++i) {
    // everywhere, beyond both ends, and at distances 1e-4 to 1e-13 of an integer or
    // half-integer index
    double ix = (1.2 * U(rng) - 0.1) * T.nb;
    if (i & 1) ix = 0.5 * std::rint(2 * ix) + (U(rng) - 0.5) * std::pow(10., -4 - 9 * U(rng));
    if (i % 16 == 1) ix = 0.5 * std::rint(2 * ix);
    const double x = lo + ix * (hi - lo) / T.nb;
    double m, L, a, m0, L0;
    const bool ok = mass_direct(T, x, m, L, a);
    const double b = mass_chain(T, x, m0, L0);
    far = std::fmax(far, std::fabs(a - b));
    err = std::fmax(err, (double)std::fabs((long double)m / std::pow(10.0L, (long double)x) - 1));
    if (!ok) continue;
    ++taken;
    wrong += (int)round(a) != (int)round(b) || (int)a != (int)b;
  }
  int special = 0;   // taken directly although not a mass
  for (double x : {(double)NAN, (double)INFINITY, -(double)INFINITY, 1e300, -1e300, 300., -400.}) {
    double m, L, a;
    special += mass_direct(T, x, m, L, a);
  }
  // the same range as wave numbers
  T.kmin = T.mmin;
  T.kmax = T.mmax;
  T.rkmin = T.rmmin;
  T.lkr = T.lmr;
  T.rlkr = T.rlmr;
  const double top = (double)T.nb * T.nb + T.nb;
  auto chain = [&](double k) {
    const double x = std::round(std::log(k / T.kmin) * T.nb / T.lkr);
    return x >= 0 ? (int)std::fmin(x, top) : (x < 0 ? (int)std::fmax(x, -1.0) : 0);
  };
  long kwrong = 0;
  for (int i = 0; i < 400000; ++i) {
    double ix = (1.5 * U(rng) - 0.2) * T.nb;
    if (i & 1) ix = 0.5 + std::rint(ix) + (U(rng) - 0.5) * std::pow(10., -4 - 11 * U(rng));
    if (i % 16 == 1) ix = 0.5 + std::floor(ix);
    const double k = T.kmin * std::exp(ix * T.lkr / T.nb);
    kwrong += kix_round(T, k) != chain(k);
  }
  for (double k : {0., -0., -1., (double)NAN, (double)INFINITY, -(double)INFINITY, 1e-300, 1e-310,
                   1e300, 1.7e308, T.kmin, T.kmax})
    kwrong += kix_round(T, k) != chain(k);
  printf("%ld %ld %.3g %.3g %d %ld\n", taken, wrong, far, err, special, kwrong);
}
