// select_wave.h -- the boundary of a Gladwell batch, found by one wave from
// error keys in its registers; shared by k_select (kernels.hip) and k_onedim.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "select_math.h"

#pragma clang fp contract(off)

namespace g3l {

__device__ __forceinline__ uint64_t readlane64(uint64_t v, int l) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l);
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ double readlane64(double v, int l) {
  return __builtin_bit_cast(double, readlane64(__builtin_bit_cast(uint64_t, v), l));
}
__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// The value of lane l + w, for lanes l < w of a wave (the others get whatever
// the permute leaves): register permutes, which take a tenth of the latency of
// a shuffle through LDS.
template <int w>
__device__ __forceinline__ uint32_t from_above32(uint32_t v) {
  if constexpr (w == 32) return __builtin_amdgcn_permlane32_swap(v, v, false, false)[1];
  else if constexpr (w == 16) return __builtin_amdgcn_permlane16_swap(v, v, false, false)[1];
  else return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x100 + w, 0xf, 0xf, true);   // row_shl
}
template <int w>
__device__ __forceinline__ uint64_t from_above(uint64_t v) {
  return ((uint64_t)from_above32<w>((uint32_t)(v >> 32)) << 32) | from_above32<w>((uint32_t)v);
}
template <int w>
__device__ __forceinline__ double from_above(double v) {
  return __builtin_bit_cast(double, from_above<w>(__builtin_bit_cast(uint64_t, v)));
}
template <int N>
struct Int {
  static constexpr int value = N;
};
// f(Int<w>) for w = 32, 16, 8, 4, 2, 1.
template <class F>
__device__ __forceinline__ void tree(F f) {
  f(Int<32>{}), f(Int<16>{}), f(Int<8>{}), f(Int<4>{}), f(Int<2>{}), f(Int<1>{});
}
__device__ __forceinline__ uint64_t wave_max(uint64_t k) {
  tree([&](auto w) {
    const uint64_t o = from_above<decltype(w)::value>(k);
    k = o > k ? o : k;
  });
  return readlane64(k, 0);
}
// Accesses of a wave to LDS that no other wave uses: a compiler barrier
// orders them.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The rounding error of t = s + e, exactly (Knuth's TwoSum).  Equal to
// Neumaier's branch on the larger operand, in fewer instructions.
__device__ __forceinline__ double sum_error(double s, double e, double t) {
  const double b = t - s;
  return (s - (t - b)) + (e - b);
}
// One step of a compensated sum (s, c) += e.
__device__ __forceinline__ void comp_add(double &s, double &c, double e) {
  const double t = s + e;
  c += sum_error(s, e, t);
  s = t;
}
// The tree of the lanes' compensated sums: lane l takes in lane l + w for
// w = 32 .. 1; lane 0 ends with the total.
__device__ __forceinline__ void comp_tree(double &s, double &c) {
  tree([&](auto w) {
    constexpr int W = decltype(w)::value;
    const double b = from_above<W>(s), cb = from_above<W>(c);
    const double t = s + b;
    c += cb + sum_error(s, b, t);
    s = t;
  });
}
__device__ __forceinline__ double comp_total(double s, double c) {
  comp_tree(s, c);
  return readlane64(s + c, 0);
}

// The converged() test of the reference on a remaining error
// (src/converged.h:10-14).
__device__ __forceinline__ bool meets(double rest, double thr) { return !(rest > 0 && rest > thr); }

// Where the batch ends: thr, the remaining error that is enough; kcap, the
// most regions the budget allows; above and below, the count of the keys
// larger and the sum of the keys smaller than those a search looks at.
struct Goal {
  double thr;
  uint64_t kcap;
  uint32_t above;
  double below;
};
// What it is: the key T of the last region popped, its multiplicity eq and the
// `take` of them that are popped, gt keys larger than T.
struct Boundary {
  uint64_t T;
  uint32_t eq, take, gt;
};

// Fewest of eq regions with key T, with gt larger keys popped before them and
// `rest` the sum of the smaller keys, that end the batch.
__device__ __forceinline__ uint32_t fewest(const Goal &g, uint64_t T, uint32_t eq, uint32_t gt,
                                           double rest) {
  const double e = __builtin_bit_cast(double, T);
  uint32_t r = eq;
  while (r > 1 && (meets(rest + (double)(eq - r + 1) * e, g.thr) || (uint64_t)gt + r - 1 >= g.kcap))
    --r;
  return r;
}

// LDS of one search.
struct SearchLds {
  uint64_t key[64];
};

template <int R>
__device__ __forceinline__ double sum_below(const uint64_t (&k)[R], uint32_t n, uint64_t T) {
  double s = 0, c = 0;
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (64u * r < n) comp_add(s, c, k[r] < T ? __builtin_bit_cast(double, k[r]) : 0.0);
  return comp_total(s, c);
}

// Boundary of the Gladwell batch (src/hcubature.cpp:971-985) over a wave's n
// keys (k[r] of lane l is entry 64 r + l, ~0 where there is none, maxkey the
// largest): regions are popped in decreasing error until the remaining error
// meets thr or kcap are popped.  Both hold for all smaller keys once they hold
// for one, so T is the largest key at which popping every key >= T is enough.
// False if it is not among these keys.
//
// A search over the keys' high words, with FP32 sums of what remains, leaves
// an interval of at most kFew keys; every lane then sums the keys below its
// own exactly.  All of it is in registers (a histogram in LDS, with its
// atomics and scans, took five times as long).  A boundary that the FP32 sums
// put outside the interval shows in the exact sums and is then found by
// bisection over the key's bits.
template <int R>
__device__ __forceinline__ bool find_boundary(const uint64_t (&k)[R], uint32_t n, uint64_t maxkey,
                                              const Goal &g, SearchLds &W, Boundary &B) {
  constexpr uint32_t kFew = 12;   // a lane's sums over them cost as much as four search steps
  const int lane = threadIdx.x & 63;
  // most often in a bisection towards a peak, only the largest goes
  if constexpr (R == 1) {
    const uint64_t largest = __ballot(lane < (int)n && k[0] == maxkey);
    if (g.above == 0 && __popcll(largest) == 1 &&
        (g.kcap == 1 || meets(g.below + sum_below(k, n, maxkey), g.thr))) {
      B = Boundary{maxkey, 1, 1, 0};
      return true;
    }
  }
  uint64_t ck = R == 1 ? k[0] : ~0ull;   // this lane's candidate
  uint32_t m = n;                        // candidates
  uint32_t above = g.above;              // keys above every candidate
  double below = g.below;                // sum of the keys below every candidate
  if (R > 1 || n > kFew) {
    // keys in units of the largest's exponent
    const int ex = -((int)(maxkey >> 52) - 1023);
    const float thr = (float)ldexp(g.thr - g.below, ex);
    float f[R];
#pragma unroll
    for (int r = 0; r < R; ++r) f[r] = (float)ldexp(__builtin_bit_cast(double, k[r]), ex);
    const uint32_t mh = (uint32_t)(maxkey >> 32);
    // whether popping every key with a high word >= t is enough; cnt: the keys
    // below
    auto enough = [&](uint32_t t, uint32_t &cnt) {
      float s = 0;
      cnt = 0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (64u * r >= n) break;
        const bool b = (uint32_t)(k[r] >> 32) < t;
        s += b ? f[r] : 0.0f;
        cnt += (uint32_t)__popcll(__ballot(b));
      }
      tree([&](auto w) {
        s += __builtin_bit_cast(float, from_above32<decltype(w)::value>(__builtin_bit_cast(uint32_t, s)));
      });
      s = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(uint32_t, s)));
      return s <= thr || (uint64_t)g.above + n - cnt >= g.kcap;
    };
    // enough at lo, not at hi: two octaves below the largest key, then four,
    // eight, ..., then halving
    uint32_t lo = 0, hi = mh + 1, nlo = 0, nhi = n, c = 0;
    for (uint32_t d = 2u << 20; d < mh && nhi - nlo > kFew; d <<= 1) {
      if (enough(mh - d, c)) {
        lo = mh - d;
        nlo = c;
        break;
      }
      hi = mh - d;
      nhi = c;
    }
    while (nhi - nlo > kFew && hi - lo > 1) {
      const uint32_t t = lo + ((hi - lo) >> 1);
      if (enough(t, c)) {
        lo = t;
        nlo = c;
      } else {
        hi = t;
        nhi = c;
      }
    }
    m = nhi - nlo;
    above += n - nhi;
    const uint64_t klo = (uint64_t)lo << 32, khi = (uint64_t)hi << 32;
    double bs = 0, bc = 0;
    uint32_t at = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (64u * r >= n) break;
      comp_add(bs, bc, k[r] < klo ? __builtin_bit_cast(double, k[r]) : 0.0);
      if (m <= 64) {
        const bool in = k[r] < khi && k[r] >= klo;
        const uint64_t bm = __ballot(in);
        if (in) W.key[at + lanes_below(bm)] = k[r];
        at += (uint32_t)__popcll(bm);
      }
    }
    below += comp_total(bs, bc);
    wave_sync();
    if (m > 64) m = 0;   // more equal high words than lanes
    ck = lane < (int)m ? W.key[lane] : ~0ull;
  }
  if (m) {
    double s = 0, c = 0;
    uint32_t eq = 0, gt = above;
    for (uint32_t j = 0; j < m; ++j) {
      const uint64_t kj = readlane64(ck, (int)j);
      comp_add(s, c, kj < ck ? __builtin_bit_cast(double, kj) : 0.0);
      eq += kj == ck;
      gt += kj > ck;
    }
    const double after = below + (s + c);
    const bool in = lane < (int)m;
    const bool mine = in && (meets(after, g.thr) || (uint64_t)gt + eq >= g.kcap);
    // enough before any candidate is popped: the boundary is further up
    const bool early = in && gt == above && above > 0 &&
                       (meets(after + (double)eq * __builtin_bit_cast(double, ck), g.thr) ||
                        above >= g.kcap);
    if (__ballot(mine) != 0 && __ballot(early) == 0) {
      const uint64_t T = wave_max(mine ? ck : 0);
      const int who = __ffsll((unsigned long long)__ballot(mine && ck == T)) - 1;
      B.T = T;
      B.eq = (uint32_t)__builtin_amdgcn_readlane((int)eq, who);
      B.gt = (uint32_t)__builtin_amdgcn_readlane((int)gt, who);
      B.take = fewest(g, T, B.eq, B.gt, readlane64(after, who));
      return true;
    }
  }
  // the largest T <= maxkey at which popping every key >= T is enough (it is a
  // key: the remaining error and the count only change just above one)
  auto enough = [&](uint64_t t, uint32_t &ge) {
    ge = g.above;
#pragma unroll
    for (int r = 0; r < R; ++r) ge += (uint32_t)__popcll(__ballot(k[r] != ~0ull && k[r] >= t));
    return ge >= g.kcap || meets(g.below + sum_below(k, n, t), g.thr);
  };
  uint32_t ge = 0;
  if (!enough(0, ge) || (g.above > 0 && enough(maxkey + 1, ge))) return false;
  uint64_t t = 0;
  for (int bit = 62; bit >= 0; --bit) {
    const uint64_t u = t | (1ull << bit);
    if (u <= maxkey && enough(u, ge)) t = u;
  }
  uint32_t eq = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) eq += (uint32_t)__popcll(__ballot(k[r] == t));
  (void)enough(t, ge);
  B.T = t;
  B.eq = eq;
  B.gt = ge - eq;
  B.take = fewest(g, t, eq, B.gt, g.below + sum_below(k, n, t));
  return true;
}

}  // namespace g3l
