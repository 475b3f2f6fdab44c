// Host build of the NFW normalisation (physics.h), ln(1 + c) and F = ln(1 + c) -
// c / (1 + c), against the expressions with the library's log, both against log1p in
// 64-bit mantissas: reads a range of c and a seed; prints the rms and the largest error
// of each logarithm in units of the last place, the rms error of each F, and how many
// of four c without a logarithm are NaN.
#include "../../g3lhalo_amd/csrc/physics.h"

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>

using namespace g3l;

int main(int argc, char **argv) {
  if (argc != 4) return 1;
  std::mt19937_64 rng(atoi(argv[3]));
  std::uniform_real_distribution<double> U(atof(argv[1]), atof(argv[2]));
  const int n = 200000;
  double max[2] = {}, sq[2] = {}, sqF[2] = {};
  for (int i = 0; i < n; ++i) {
    const double c = U(rng), l = std::log(1. + c);
    const long double w = log1pl((long double)c), wF = w - (long double)c / (1 + (long double)c);
    double lc, F;
    P64::nfw_norm(c, lc, F);
    const double v[2] = {lc, l}, vF[2] = {F, l - c / (1. + c)};
    for (int j = 0; j < 2; ++j) {
      const double e = (double)std::fabs((v[j] - w) / std::ldexp(1.L, std::ilogb((double)w) - 52));
      const double eF =
          (double)std::fabs((vF[j] - wF) / std::ldexp(1.L, std::ilogb((double)wF) - 52));
      max[j] = std::fmax(max[j], e);
      sq[j] += e * e;
      sqF[j] += eF * eF;
    }
  }
  printf("%.6g %.6g %.6g %.6g %.6g %.6g\n", std::sqrt(sq[0] / n), max[0], std::sqrt(sq[1] / n),
         max[1], std::sqrt(sqF[0] / n), std::sqrt(sqF[1] / n));
  int nan = 0;
  for (double c : {-1., -1.5, (double)NAN, -(double)INFINITY}) {
    double lc, F;
    P64::nfw_norm(c, lc, F);
    nan += std::isnan(lc) && std::isnan(F);
  }
  printf("%d\n", nan);
}
