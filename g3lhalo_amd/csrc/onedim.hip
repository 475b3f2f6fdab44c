// onedim.hip -- k_onedim: whole adaptive 1-D integrals in one kernel.
//
// The integrals (n_bar(z), and the precomputation's sigma^2 and distances) are
// many and small: an n_bar integral ends with about 600 regions after 26
// rounds, a sigma^2 integral with about 50 after 45.  Run as rounds of the
// general engine (an evaluation, a selection and a counter copy per round) one
// HOD set took 3.7 ms, nearly all of it launches, host turns and the fixed
// cost of the selection blocks; 256 sets took 104 ms and the 65,000 integrals
// of a 128-bin precomputation 118 ms.
//
// Here a block refines up to eight integrals from root to convergence, one
// wave per integral, in lockstep rounds:
//   select    each wave: totals, stop test, Gladwell batch (the semantics of
//             k_select, src/hcubature.cpp:938-989);
//   evaluate  the whole block: the abscissa-only part of the integrand at the
//             15 points of every region that it has not met before;
//   reduce    the whole block: the new regions' rule sums from those values.
// The integrals of a group share their box, so their regions are nodes of one
// bisection tree and mostly the same ones (n_bar's integrand jumps at the same
// mass bins at every redshift): a node's masses, table indices and HOD
// occupations, most of an n_bar point's work, are computed once for all the
// integrals a block takes from one group.  Point values are the same
// expressions in the same order whichever integral asked first.
//
// Measured: one HOD set (256 integrals) 3.7 -> 1.35 ms, 256 sets 104 -> 35 ms,
// the precomputation 118 -> 14 ms.  What is left is instruction issue and the
// latency of the selection, whose waves are alone with their integrals.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "onedim.h"
#include "rules.h"
#include "select_math.h"

#pragma clang fp contract(off)

namespace g3l {

namespace {

constexpr int kThreads = 512, kWaves = kThreads / 64;
static_assert(kWaves == kOneDimMaxUnit, "one wave per integral of a unit");
constexpr int kPts = 15;
constexpr uint32_t kMaxSplit = kOneDimCap / 2;   // regions cut in one round
constexpr uint32_t kChunk = 32;                  // regions reduced together (precomputation)
static_assert(kChunk * kPts <= kThreads, "a point per thread");

// Device memory of a block.  Node values are field-major so that the lanes of
// a wave, which reduce neighbouring nodes, read neighbouring words.
struct Store {
  double2 ab[kPts][kOneDimNodes];
  int32_t ix[kPts][kOneDimNodes];
  double c[kOneDimNodes], h[kOneDimNodes];
  // regions of each wave's integral: rule value, error, node
  double val[kWaves][kOneDimCap], err[kWaves][kOneDimCap];
  uint16_t node[kWaves][kOneDimCap];
};

struct WaveLds {
  // selection: 64 bins of fixed-point error sums and counts
  unsigned long long sum[64];
  uint32_t cnt[64];
  uint64_t key[64];        // keys of the boundary bin
  uint16_t split[kMaxSplit];
};

struct Lds {
  WaveLds w[kWaves];
  uint32_t child[kOneDimNodes];        // first of a node's two children, 0: none
  uint16_t fresh[kOneDimNodes / 2];    // nodes split for the first time this round
  double f[kChunk * kPts];             // point values (precomputation)
  uint32_t nnodes, nfresh, full;
  uint32_t n[kWaves], cut[kWaves];     // regions, and regions cut this round, per integral
  int32_t row[kWaves];                 // hmf row of each integral's redshift (n_bar)
  OneDimJob job[kWaves];
};
// Dynamic LDS, so that the functions kept out of line address it as LDS.
extern __shared__ __align__(16) unsigned char lds_raw[];
__device__ __forceinline__ Lds &lds() { return *reinterpret_cast<Lds *>(lds_raw); }

// The part of the integrand that depends on the abscissa alone.
//   n_bar: ab = (m, Ncen + Nsat), ix = the mass index;
//   sigma^2, d sigma^2/dm: ab = (amplitude T(k)^2, k^ns);
//   distance, amplitude: ab.x = the integrand (one integral per group).
template <bool PRE>
__device__ __forceinline__ void one_dim_node(const DevTables &T, const OneDimGroup &g, double t1,
                                             double x, double2 &ab, int32_t &ix) {
  if constexpr (!PRE) {
    TermArgs a{};
    a.h1 = g.h;
    const Mass M = make_mass<P64R>(T, x, 0);
    const Occ o = occ1<P64R>(a, M);
    ab = double2{M.m, o.nc + o.ns};
    ix = M.ir;
  } else {
    const PrecompParams &p = *reinterpret_cast<const PrecompParams *>(g.aux);
    ix = 0;
    if (g.mode == kOneDComoving) {
      ab = double2{precomp_distance(p, x), 0.0};
    } else if (g.mode == kOneDAmplitude) {
      ab = double2{precomp_amplitude(p, x, t1), 0.0};
    } else {
      const double t = eh_transfer(p, x);
      ab = double2{p.amplitude * t * t, pow(x, p.ns)};
    }
  }
}

// The integrand of one integral from its node values.
__device__ __forceinline__ double precomp_point(int mode, const OneDimJob &j, double x,
                                                const double2 &ab) {
  if (mode == kOneDComoving || mode == kOneDAmplitude) return ab.x;
  const double spectrum = ab.x * j.t2 * j.t2 * ab.y;   // eh_spectrum's order
  const double W = tophat(x, j.t1);
  if (mode == kOneDSigma2) return x * x * W * W * spectrum;
  return x * x * W * d_tophat(x, j.t1) * j.t3 * spectrum;
}

__device__ __forceinline__ double lane0(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
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
  return __builtin_bit_cast(uint64_t, lane0(__builtin_bit_cast(double, k)));
}
// The LDS of a wave is its own: a compiler barrier orders its accesses.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// One Neumaier step (s, c) += e.
__device__ __forceinline__ void comp_add(double &s, double &c, double e) {
  const double t = s + e;
  c += fabs(s) >= fabs(e) ? (s - t) + e : (e - t) + s;
  s = t;
}
// Lane 0's tree sum of the lanes' (s, c), in every lane.
__device__ __forceinline__ double comp_total(double s, double c) {
  tree([&](auto w) {
    constexpr int W = decltype(w)::value;
    const double b = from_above<W>(s), cb = from_above<W>(c);
    const double t = s + b;
    c += cb + (fabs(s) >= fabs(b) ? (s - t) + b : (b - t) + s);
    s = t;
  });
  return lane0(s + c);
}

// The converged() test of the reference on a remaining error.
__device__ __forceinline__ bool meets(double rest, double thr) { return !(rest > 0 && rest > thr); }

// Sum of the keys below T, compensated, over a wave's R x 64 keys (~0: none).
template <int R>
__device__ __forceinline__ double sum_below(const uint64_t (&k)[R], uint32_t n, uint64_t T) {
  double s = 0, c = 0;
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (64u * r < n) comp_add(s, c, k[r] < T ? __builtin_bit_cast(double, k[r]) : 0.0);
  return comp_total(s, c);
}

// Boundary of the Gladwell batch over n keys (k[r] of lane l is slot 64 r + l,
// ~0 where there is none): the key T of the last region popped and how many
// regions with that key are popped, such that the count is the first at which
// the remaining error meets thr.  The remaining error after popping every key
// >= T falls with T, so T is the largest key at which it meets thr.
//
// At most 64 regions: every lane sums the keys below its own.  More: a
// histogram of the keys' distance below the largest (two bins per octave,
// exact fixed-point sums) names the bin that holds the boundary, narrowed
// until at most 64 keys are left, whose lanes do the same; a boundary that the
// truncated sums put into the wrong bin shows in the exact sums and is then
// found by bisection over the key's bits.
template <int R>
__device__ __forceinline__ void find_boundary(const uint64_t (&k)[R], uint32_t n, uint64_t maxkey,
                                              double thr, WaveLds &W, uint64_t &T, uint32_t &take) {
  const int lane = threadIdx.x & 63;
  uint64_t ck = ~0ull;      // this lane's candidate
  uint32_t m = 0;           // candidates
  double below = 0;         // sum of the keys below every candidate
  bool found = false, top = true;
  if constexpr (R == 1) {
    // most often only the largest goes (the bisection towards a peak)
    const uint64_t largest = __ballot(lane < (int)n && k[0] == maxkey);
    if (__popcll(largest) == 1 && meets(sum_below(k, n, maxkey), thr)) {
      T = maxkey;
      take = 1;
      return;
    }
    ck = k[0];
    m = n;
  } else {
    const int shift = sel_shift(maxkey, n);
    const double thr_fx = ldexp(thr, shift);
    // candidates: distance d = maxkey - key in [lo, lo + width)
    uint64_t lo = 0, width = 1ull << 63;
    int s = 51;
    unsigned long long rest_after = 0;  // fixed-point sum of the keys beyond the range
    for (;;) {
      W.sum[lane] = 0;
      W.cnt[lane] = 0;
      wave_sync();
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (64u * r >= n) break;
        const uint64_t d = maxkey - k[r] - lo;   // absent keys wrap to >= 2^63
        if (k[r] <= maxkey && k[r] <= maxkey - lo && d < width) {
          const uint64_t q = d >> s;
          const int b = q < 63 ? (int)q : 63;
          atomicAdd(&W.cnt[b], 1u);
          atomicAdd(&W.sum[b], fixed_err(k[r], shift));
        }
      }
      wave_sync();
      // suffix sums: what remains in the range beyond bin `lane`
      const unsigned long long own = W.sum[lane];
      unsigned long long suf = own;
#pragma unroll
      for (int w = 1; w < 64; w <<= 1) {
        const uint32_t l2 = __shfl_down((uint32_t)suf, w), h2 = __shfl_down((uint32_t)(suf >> 32), w);
        if (lane + w < 64) suf += ((unsigned long long)h2 << 32) | l2;
      }
      const unsigned long long rest = suf - own + rest_after;
      const uint64_t hit = __ballot((double)rest <= thr_fx && W.cnt[lane] != 0);
      int b = hit ? __ffsll((unsigned long long)hit) - 1
                  : 63 - __clzll((long long)__ballot(W.cnt[lane] != 0));
      b = __builtin_amdgcn_readfirstlane(b);
      m = (uint32_t)__builtin_amdgcn_readlane((int)W.cnt[lane], b);
      {
        const uint32_t rl = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)rest, b);
        const uint32_t rh = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(rest >> 32), b);
        rest_after = ((unsigned long long)rh << 32) | rl;
      }
      lo += (uint64_t)b << s;
      width = b == 63 ? width - ((uint64_t)63 << s) : 1ull << s;
      if (m <= 64 || width <= 1) break;
      s = 58 - __clzll((long long)(width - 1));   // ceil(log2 width) - 6
      s = s < 0 ? 0 : s;
    }
    top = lo == 0;
    const uint64_t kmin = maxkey - lo >= width - 1 ? maxkey - lo - (width - 1) : 0;
    below = sum_below(k, n, kmin);
    if (m > 64) {   // one key, many regions
      T = maxkey - lo;
      uint32_t eq = m;
      const double kt = __builtin_bit_cast(double, T);
      found = meets(below, thr) && (top || !meets(below + (double)eq * kt, thr));
      if (found) {
        while (eq > 1 && meets(below + (double)(m - eq + 1) * kt, thr)) --eq;
        take = eq;
        return;
      }
    } else {
      uint32_t at = 0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (64u * r >= n) break;
        const bool in = k[r] <= maxkey - lo && k[r] >= kmin;
        const uint64_t bm = __ballot(in);
        if (in) W.key[at + lanes_below(bm)] = k[r];
        at += (uint32_t)__popcll(bm);
      }
      wave_sync();
      ck = lane < (int)m ? W.key[lane] : ~0ull;
    }
  }
  if (m <= 64) {
    double s = 0, c = 0, all = 0, allc = 0;
    uint32_t eq = 0;
    for (uint32_t j = 0; j < m; ++j) {
      const uint32_t jl = __builtin_amdgcn_readlane((int)(uint32_t)ck, j);
      const uint32_t jh = __builtin_amdgcn_readlane((int)(uint32_t)(ck >> 32), j);
      const uint64_t kj = ((uint64_t)jh << 32) | jl;
      const double e = __builtin_bit_cast(double, kj);
      comp_add(s, c, kj < ck ? e : 0.0);
      eq += kj == ck;
      if constexpr (R > 1) comp_add(all, allc, e);
    }
    const double after = below + (s + c);
    const bool mine = lane < (int)m && meets(after, thr);
    const bool early = !top && meets(below + (all + allc), thr);   // met before this bin
    if (__ballot(mine) != 0 && !early) {
      T = wave_max(mine ? ck : 0);
      const int who = __ffsll((unsigned long long)__ballot(mine && ck == T)) - 1;
      const uint32_t cntT = (uint32_t)__builtin_amdgcn_readlane((int)eq, who);
      const uint64_t ab = __builtin_bit_cast(uint64_t, after);
      const uint32_t al = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)ab, who);
      const uint32_t ah = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(ab >> 32), who);
      const double rest = __builtin_bit_cast(double, ((uint64_t)ah << 32) | al);
      uint32_t r = cntT;
      while (r > 1 && meets(rest + (double)(cntT - r + 1) * __builtin_bit_cast(double, T), thr)) --r;
      take = r;
      return;
    }
  }
  // the largest T <= maxkey at which the keys below T meet thr (it is a key:
  // the sum only changes just above one)
  uint64_t t = 0;
  for (int bit = 62; bit >= 0; --bit) {
    const uint64_t u = t | (1ull << bit);
    if (u <= maxkey && meets(sum_below(k, n, u), thr)) t = u;
  }
  uint32_t eq = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) eq += (uint32_t)__popcll(__ballot(k[r] == t));
  const double rest = sum_below(k, n, t);
  uint32_t r = eq;
  while (r > 1 && meets(rest + (double)(eq - r + 1) * __builtin_bit_cast(double, t), thr)) --r;
  T = t;
  take = r;
}

// One integral's state; every field is the same in all lanes of its wave.
struct WaveState {
  uint32_t n, flags, K;
  double V;
};

// Totals, stop test and batch of one integral's n <= 64 R regions.  Sets
// st.flags when it ends, otherwise st.K and the batch in W.split.
//
// The totals keep the order they have in k_select, whose 256 threads take the
// slots in strides and then add pairwise: lane l holds the threads l, l + 64,
// l + 128 and l + 192.
template <int R>
__device__ __noinline__ void wave_round(const double *val, const double *err, double reltol,
                                    WaveState &st) {
  const int lane = threadIdx.x & 63;
  WaveLds &W = lds().w[threadIdx.x >> 6];
  const uint32_t n = st.n;
  constexpr int V4 = R < 4 ? R : 4;
  constexpr int B = R < 8 ? R : 8;   // loads in flight per array
  uint64_t k[R];
  double vs[V4] = {}, vc[V4] = {}, es[V4] = {};
  bool bad = false;
  uint64_t maxkey = 0;
#pragma unroll
  for (int r0 = 0; r0 < R; r0 += B) {
    double v[B], e[B];
#pragma unroll
    for (int r = 0; r < B; ++r) {
      const uint32_t i = 64 * (r0 + r) + lane;
      v[r] = i < n ? val[i] : 0.0;
      e[r] = i < n ? err[i] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < B; ++r) {
      bad |= !isfinite(v[r]) || !isfinite(e[r]);
      comp_add(vs[r & (V4 - 1)], vc[r & (V4 - 1)], v[r]);
      es[r & (V4 - 1)] += e[r];
      const uint64_t ke = err_key(e[r]);   // 0 where there is no region
      k[r0 + r] = 64u * (r0 + r) + lane < n ? ke : ~0ull;
      maxkey = ke > maxkey ? ke : maxkey;
    }
  }
#pragma unroll
  for (int w = V4 / 2; w > 0; w >>= 1) {
#pragma unroll
    for (int q = 0; q < w; ++q) {
      const double a = vs[q], b = vs[q + w], t = a + b;
      vc[q] += vc[q + w] + (fabs(a) >= fabs(b) ? (a - t) + b : (b - t) + a);
      vs[q] = t;
      es[q] += es[q + w];
    }
  }
  const double V = comp_total(vs[0], vc[0]);
  double E = es[0];
  tree([&](auto w) { E += from_above<decltype(w)::value>(E); });
  E = lane0(E);
  st.V = V;
  st.K = 0;
  if (__ballot(bad) != 0) st.flags |= kJobNonfinite;
  const double thr = fabs(V) * reltol;
  if (!(E > 0 && E > thr)) {
    st.flags |= kJobDone | kJobConverged;
    return;
  }
  maxkey = wave_max(maxkey);
  uint64_t T = 0;
  uint32_t take = 0;
  find_boundary<R>(k, n, maxkey, thr, W, T, take);
  // regions above T and the first `take` of those at T, in slot order
  uint32_t ties = 0, K = 0;
  uint32_t sel = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (64u * r >= n) break;
    const bool in = k[r] != ~0ull, tie = in && k[r] == T;
    const uint64_t tm = __ballot(tie);
    const bool s = in && (k[r] > T || (tie && ties + lanes_below(tm) < take));
    ties += (uint32_t)__popcll(tm);
    sel |= s ? 1u << r : 0u;
    K += (uint32_t)__popcll(__ballot(s));
  }
  if (n + K > kOneDimCap) {
    st.flags |= kJobDone | kJobPoolFull;
    return;
  }
  st.K = K;
  uint32_t at = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (64u * r >= n) break;
    const bool s = sel >> r & 1u;
    const uint64_t sm = __ballot(s);
    if (s) W.split[at + lanes_below(sm)] = (uint16_t)(64 * r + lane);
    at += (uint32_t)__popcll(sm);
  }
}

// One round of this wave's integral, by the number of its regions, and the
// nodes its batch needs: the first wave to split a node makes its children.
__device__ __forceinline__ void wave_select(const double *val, const double *err,
                                            const uint16_t *node, double reltol, WaveState &st) {
  if (st.n <= 64) wave_round<1>(val, err, reltol, st);
  else if (st.n <= 256) wave_round<4>(val, err, reltol, st);
  else if (st.n <= 1024) wave_round<16>(val, err, reltol, st);
  else wave_round<32>(val, err, reltol, st);
  Lds &S = lds();
  const WaveLds &W = S.w[threadIdx.x >> 6];
  wave_sync();
  for (uint32_t a = threadIdx.x & 63; a < st.K; a += 64) {
    const uint32_t v = node[W.split[a]];
    if (atomicCAS(&S.child[v], 0u, ~0u) == 0u) {
      const uint32_t id = atomicAdd(&S.nnodes, 2u);
      if (id + 2 <= kOneDimNodes) {
        S.child[id] = 0;
        S.child[id + 1] = 0;
        S.child[v] = id;
        S.fresh[atomicAdd(&S.nfresh, 1u)] = (uint16_t)v;
      } else {
        S.child[v] = 0;
        S.full = 1;
      }
    }
  }
}

// Region i of the block's round: the integral it belongs to (w), its node and
// its slot.  An integral's regions are the left (even) and right (odd) halves
// of those in its W.split; the left half keeps its parent's slot, the right
// one takes the next free slot.
__device__ __forceinline__ void place(const Store &G, uint32_t i, bool root, uint32_t &w,
                                      uint32_t &id, uint32_t &slot) {
  const Lds &S = lds();
  w = 0;
  if (root) {
    w = i;
    id = 0;
    slot = 0;
    return;
  }
  uint32_t at = 0;
#pragma unroll
  for (int q = 0; q < kWaves - 1; ++q) {
    const uint32_t next = at + 2 * S.cut[q];
    if (i >= next && w == (uint32_t)q) {
      ++w;
      at = next;
    }
  }
  const uint32_t r = i - at, p = S.w[w].split[r >> 1];
  id = S.child[G.node[w][p]] + (r & 1u);
  slot = (r & 1u) ? S.n[w] + (r >> 1) : p;
}

// Rule sums of the `total` regions of the block's round (place), or of the
// root of each of `total` integrals.  Every thread of the block calls it.
template <bool PRE>
__device__ __forceinline__ void block_reduce(const OneDimLaunch &L, int mode, Store &G,
                                             uint32_t total, bool root) {
  Lds &S = lds();
  const uint32_t tid = threadIdx.x;
  if constexpr (!PRE) {
    // a region per thread: a point is two loads, a table look-up and two products
    for (uint32_t i = tid; i < total; i += kThreads) {
      uint32_t w, id, slot;
      place(G, i, root, w, id, slot);
      const double *hmf = L.T.hmf + S.row[w];
      double f[kPts], v, e;
#pragma unroll
      for (int j = 0; j < kPts; ++j) {
        const double2 ab = G.ab[j][id];
        f[j] = ab.x * hmf[G.ix[j][id]] * ab.y;
      }
      gk_reduce(f, G.h[id], v, e);
      G.val[w][slot] = v;
      G.err[w][slot] = e;
      G.node[w][slot] = (uint16_t)id;
    }
  } else {
    // a point per thread: a point takes the window's sin and cos of a large
    // argument, and in most rounds every integral has two regions
    for (uint32_t i0 = 0; i0 < total; i0 += kChunk) {
      const uint32_t q = tid / kPts, i = i0 + q, j = tid - kPts * q;
      if (q < kChunk && i < total) {
        uint32_t w, id, slot;
        place(G, i, root, w, id, slot);
        const double c = G.c[id], h = G.h[id];
        double x;
        rule_point<1>((int)j, &c, &h, &x);
        S.f[tid] = precomp_point(mode, S.job[w], x, G.ab[j][id]);
      }
      __syncthreads();
      if (tid < kChunk && i0 + tid < total) {
        uint32_t w, id, slot;
        place(G, i0 + tid, root, w, id, slot);
        double v, e;
        gk_reduce(S.f + kPts * tid, G.h[id], v, e);
        G.val[w][slot] = v;
        G.err[w][slot] = e;
        G.node[w][slot] = (uint16_t)id;
      }
      __syncthreads();
    }
  }
}

}  // namespace

// Four waves per SIMD: two blocks per compute unit, one block's barriers and
// serial stretches beside the other's work.
template <bool PRE>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_onedim(
    OneDimLaunch L) {
  Lds &S = lds();
  Store &G = reinterpret_cast<Store *>(L.store)[blockIdx.x];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // a block takes consecutive units, whose integrals mostly share one group,
  // and keeps the nodes as long as the group stays
  const uint32_t u0 = (uint32_t)((uint64_t)L.nunits * blockIdx.x / gridDim.x);
  const uint32_t u1 = (uint32_t)((uint64_t)L.nunits * (blockIdx.x + 1) / gridDim.x);
  uint32_t have = ~0u;   // group whose nodes the block holds
  for (uint32_t u = u0; u < u1;) {
    const OneDimUnit U = L.units[u];
    const OneDimGroup &g = L.groups[U.group];
    const bool mine = wave < (int)U.count;
    __syncthreads();   // the previous unit's LDS is done with
    const bool reuse = have == U.group && S.nnodes <= kOneDimNodes / 2;
    const double t1 = L.jobs[g.job0 + U.first].t1;
    if (tid < (int)U.count) {
      const OneDimJob job = L.jobs[g.job0 + U.first + tid];
      S.job[tid] = job;
      if constexpr (!PRE) S.row[tid] = zix_round(L.T, job.t1) * L.T.nb;
    }
    __syncthreads();
    if (!reuse) {
      if (tid == 0) {
        S.nnodes = 1;
        S.child[0] = 0;
        G.c[0] = 0.5 * (g.lo + g.hi);
        G.h[0] = 0.5 * (g.hi - g.lo);
      }
      if (tid < kPts) {
        const double c = 0.5 * (g.lo + g.hi), h = 0.5 * (g.hi - g.lo);
        double x;
        rule_point<1>(tid, &c, &h, &x);
        one_dim_node<PRE>(L.T, g, t1, x, G.ab[tid][0], G.ix[tid][0]);
      }
    }
    if (tid == 0) S.full = 0;
    __syncthreads();
    WaveState st{1, mine ? 0u : (uint32_t)kJobDone, 0, 0.0};
    block_reduce<PRE>(L, g.mode, G, U.count, true);
    bool again = false;
    for (;;) {
      if (tid == 0) S.nfresh = 0;
      __syncthreads();
      st.K = 0;
      if (!(st.flags & kJobDone)) wave_select(G.val[wave], G.err[wave], G.node[wave], L.reltol, st);
      if (lane == 0) {
        S.n[wave] = st.n;
        S.cut[wave] = st.K;
      }
      __syncthreads();
      uint32_t total = 0;
#pragma unroll
      for (int q = 0; q < kWaves; ++q) total += 2 * S.cut[q];
      if (S.full) {
        // out of nodes: from the start with an empty tree; or, if it was
        // empty, its integrals one by one
        again = reuse;
        break;
      }
      if (total == 0) break;
      const uint32_t np = 2 * kPts * S.nfresh;
      for (uint32_t i = tid; i < np; i += kThreads) {
        const uint32_t pr = i / (2 * kPts), r = i - pr * 2 * kPts;
        const uint32_t right = r >= kPts ? 1u : 0u;
        const int j = (int)(r - right * kPts);
        const uint32_t v = S.fresh[pr], id = S.child[v] + right;
        // the halves of a split, as in the cut of src/hcubature.cpp:206-218
        const double h = G.h[v] * 0.5, c = right ? G.c[v] + h : G.c[v] - h;
        double x;
        rule_point<1>(j, &c, &h, &x);
        one_dim_node<PRE>(L.T, g, t1, x, G.ab[j][id], G.ix[j][id]);
        if (j == 0) {
          G.c[id] = c;
          G.h[id] = h;
        }
      }
      if (np) __syncthreads();
      block_reduce<PRE>(L, g.mode, G, total, false);
      st.n += st.K;
    }
    have = again ? ~0u : U.group;
    if (again) continue;
    ++u;
    if (mine && lane == 0) {
      const uint32_t i = U.first + wave;
      if (!(st.flags & kJobDone)) {
        L.retry[atomicAdd(L.nretry, 1u)] = OneDimUnit{U.group, i, 1};
      } else {
        g.out[i] = L.scale * st.V;
        if (st.flags & (kJobPoolFull | kJobNonfinite))
          atomicMin(L.failed, ((unsigned long long)U.group << 40) | ((unsigned long long)i << 8) |
                                  st.flags);
      }
    }
  }
}

size_t one_dim_store_bytes() { return (sizeof(Store) + 255) / 256 * 256; }
int one_dim_blocks_per_cu() { return 2; }

template <bool PRE>
static hipError_t launch(const OneDimLaunch &L, uint32_t blocks, hipStream_t s) {
  // more than 64 KB of dynamic LDS has to be asked for
  const hipError_t e =
      hipFuncSetAttribute(reinterpret_cast<const void *>(&k_onedim<PRE>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(Lds));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_onedim<PRE>), dim3(blocks), dim3(kThreads), sizeof(Lds), s, L);
  return hipGetLastError();
}

hipError_t launch_one_dim(bool precomp, const OneDimLaunch &L, uint32_t blocks, hipStream_t s) {
  if (L.nunits == 0) return hipSuccess;
  if (blocks == 0 || blocks > L.nunits) return hipErrorInvalidValue;
  return precomp ? launch<true>(L, blocks, s) : launch<false>(L, blocks, s);
}

}  // namespace g3l
