// The boundary of a Gladwell batch as one wave finds it (find_boundary of
// select_wave.h, run on the host lane by lane) against popping the sorted keys one by
// one: reads a seed; prints the searches made, those that found another boundary, and
// those with a boundary outside the given keys that did not say so.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <random>
#include <vector>

#include "../../g3lhalo_amd/csrc/select_wave.h"

using namespace g3l;

struct Search {
  std::vector<uint64_t> keys;
  Goal g;
};
static const Search *job;
static int width;          // keys per lane
static SearchLds W;
static Boundary got[64];
static bool ok[64];

template <int R>
static void lane_search() {
  const int l = hostwave::lane;
  const uint32_t n = (uint32_t)job->keys.size();
  uint64_t k[R], m = 0;
  for (int r = 0; r < R; ++r) {
    const uint32_t i = 64 * r + l;
    k[r] = i < n ? job->keys[i] : ~0ull;
    if (i < n && k[r] > m) m = k[r];
  }
  ok[l] = find_boundary<R>(k, n, wave_max(m), job->g, W, got[l]);
}
static void search() {
  hostwave::run(width == 1    ? lane_search<1>
                : width == 4  ? lane_search<4>
                : width == 16 ? lane_search<16>
                              : lane_search<32>);
}

static double value(uint64_t k) { return __builtin_bit_cast(double, k); }
static long searches = 0, wrong = 0, silent = 0;

// keys: all of an integral's; a search among those of ranks [first, last) of them
static void check(std::vector<uint64_t> keys, double thr, uint64_t kcap, size_t first, size_t last) {
  std::sort(keys.begin(), keys.end(), std::greater<uint64_t>());
  // what remains after the first i have been popped, smallest first
  std::vector<double> rest(keys.size() + 1, 0.0);
  for (size_t i = keys.size(); i-- > 0;) rest[i] = rest[i + 1] + value(keys[i]);
  size_t K = 0;
  do ++K;
  while (K < keys.size() && !(meets(rest[K], thr) || K >= kcap));
  Boundary want{};
  want.T = keys[K - 1];
  for (size_t i = 0; i < keys.size(); ++i) {
    want.eq += keys[i] == want.T;
    want.gt += keys[i] > want.T;
  }
  want.take = (uint32_t)K - want.gt;
  Search s;
  s.keys.assign(keys.begin() + first, keys.begin() + last);
  std::shuffle(s.keys.begin(), s.keys.end(), std::mt19937(first + keys.size()));
  s.g = Goal{thr, kcap, (uint32_t)first, rest[last]};
  const size_t n = last - first;
  width = n <= 64 ? 1 : n <= 256 ? 4 : n <= 1024 ? 16 : 32;
  job = &s;
  search();
  ++searches;
  const bool among = want.gt >= first && want.gt + want.eq <= last;
  for (int l = 0; l < 64; ++l) {
    if (!among) {
      if (ok[l]) {
        ++silent;
        printf("n %zu of %zu from %zu kcap %llu: not among them\n", n, keys.size(), first,
               (unsigned long long)kcap);
        return;
      }
    } else if (!ok[l] || got[l].T != want.T || got[l].eq != want.eq || got[l].take != want.take ||
               got[l].gt != want.gt) {
      ++wrong;
      printf("n %zu of %zu from %zu kcap %llu thr %g lane %d: %d T %g eq %u take %u gt %u, want %g "
             "%u %u %u\n", n, keys.size(), first, (unsigned long long)kcap, thr, l, (int)ok[l],
             value(got[l].T), got[l].eq, got[l].take, got[l].gt, value(want.T), want.eq, want.take,
             want.gt);
      return;
    }
  }
}

// All of the keys, and the ranges of equal keys around and beside the boundary, as a
// histogram bin would hold them.
static void checks(const std::vector<uint64_t> &keys, double thr, uint64_t kcap, std::mt19937_64 &rng) {
  const size_t n = keys.size();
  check(keys, thr, kcap, 0, n);
  std::vector<uint64_t> s = keys;
  std::sort(s.begin(), s.end(), std::greater<uint64_t>());
  for (int i = 0; i < 2; ++i) {
    size_t a = rng() % n, b = a + 1 + rng() % (n - a);
    while (a > 0 && s[a - 1] == s[a]) --a;
    while (b < n && s[b] == s[b - 1]) ++b;
    check(keys, thr, kcap, a, b);
  }
}

int main(int argc, char **argv) {
  if (argc != 2) return 1;
  std::mt19937_64 rng(atoi(argv[1]));
  auto uni = [&] { return (double)(rng() >> 11) * 0x1p-53; };
  for (uint32_t n : {1u, 2u, 11u, 13u, 63u, 64u, 65u, 200u, 256u, 257u, 1000u, 1024u, 1500u, 2048u})
    for (int kind = 0; kind < 6; ++kind) {
      std::vector<uint64_t> keys(n);
      for (uint32_t i = 0; i < n; ++i) {
        double e = 1;
        switch (kind) {
          case 0: e = 0.75; break;                                      // all equal
          case 1: e = std::ldexp(1 + uni(), -(int)(300 * uni())); break;   // 300 octaves
          case 2: e = std::floor(1 + 0x1p30 * uni()); break;            // whole numbers
          case 3: e = std::floor(4 * uni()); break;                     // a few, and zeros
          case 4: e = 0x1p40 + std::floor(0x1p10 * uni()); break;       // equal high words
          default: e = std::ldexp(uni(), -1022); break;                 // denormal
        }
        keys[i] = err_key(e);
      }
      if (kind == 3) keys[0] = err_key(3);
      double total = 0;
      std::vector<uint64_t> s = keys;
      std::sort(s.begin(), s.end());
      // sums of the smallest keys: a threshold at one, a unit beside it (whole numbers:
      // within the rounding of a 32-bit sum), none and all
      std::vector<double> below(n + 1, 0.0);
      for (uint32_t i = 0; i < n; ++i) below[i + 1] = below[i] + value(s[i]);
      total = below[n];
      const uint32_t at = (uint32_t)(rng() % (n + 1));
      std::vector<double> thrs = {0.0, 0.5 * total, 2 * total};
      if (kind == 2 || kind == 3 || kind == 4)   // sums of whole numbers are exact
        thrs.insert(thrs.end(), {below[at], below[at] + 1, below[at] - 1});
      for (double thr : thrs) checks(keys, thr, ~0ull, rng);
      for (uint64_t kcap : {(uint64_t)1, (uint64_t)(n + 1) / 2, (uint64_t)n})
        checks(keys, 1e-3 * total, kcap, rng);
    }
  printf("%ld %ld %ld\n", searches, wrong, silent);
  return 0;
}
