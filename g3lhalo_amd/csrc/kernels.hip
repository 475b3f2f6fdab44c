// kernels.hip -- gfx950 kernels of the adaptive cubature engine.
//
//   k_eval<KIND>   fused: generate the rule points of a group of regions,
//                  evaluate the integrand, reduce each region to (value,
//                  error, split dimension) from LDS.  The hot kernel.
//   k_roots        one root region per integral (src/hcubature.cpp:160-172).
//   k_select       per integral and refinement round: totals, convergence,
//                  Gladwell batch selection and region cuts
//                  (src/hcubature.cpp:938-989), appending the children to
//                  the evaluation lists.
//   k_zero         clears the round counters (a kernel rather than a memset
//                  so the round can be captured in a graph).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"
#include "physics.h"
#include "rules.h"
#include "select_math.h"
#include "select_wave.h"

#pragma clang fp contract(off)

namespace g3l {

// Most integrals for which k_select takes 1024 threads each; the blocks of more
// hide one another's latency better at 256.  Selection time of a whole run at
// 256 / 1024 threads: 9 integrals of 5e6 evaluations 1.43 / 1.11 ms, 411 2.06 /
// 1.80, 1650 5.16 / 4.68; 1500 of 2e5 evaluations 1.03 / 1.15, 9000 of 1e6
// 7.12 / 8.72.
constexpr uint32_t kSelectWideJobs = 512;

// ------------------------------------------------------------ evaluation
template <int KIND, class P>
__device__ __forceinline__ double integrand(const DevTables &T, const TermArgs &a,
                                            const double *x) {
  using Q = typename EvalPolicy<KIND, P>::type;
  if constexpr (KIND == kNbar) {
    return nbar_kernel<Q>(T, a, x);
  } else {
    DirectSrc<KIND, Q> s(T, a, x);
    return integrand_src<KIND, Q>(T, a, s);
  }
}

// Launch variants: a kernel template parameter KIND carries the integrand
// kind in its low four bits and a block-shape variant above them; kind_of_kv
// and variant_of_kv take it apart.  Every variant computes the same values.
constexpr int kVariantShift = 4;
constexpr int kNumVariants = 4;
__host__ __device__ constexpr int kind_of_kv(int kv) { return kv & ((1 << kVariantShift) - 1); }
__host__ __device__ constexpr int variant_of_kv(int kv) { return kv >> kVariantShift; }
__host__ __device__ constexpr int make_kv(int kind, int v) { return kind | (v << kVariantShift); }

// G regions per block and NT threads: every pass gives each thread one
// item per round, in straight-line code -- no loop for the compiler to hoist
// the FP64 constants of the special functions out of, which otherwise pins
// them in registers for the whole kernel and drops occupancy to one wave per
// SIMD.  Four shapes per dimension, picked per kind at run time
// (g3l_autotune): variant 0 fills one block of up to 1024 threads, variants
// 1 and 2 take fewer regions so that more blocks share a compute unit and
// one block's barriers overlap another's work, and variant 3 is a group
// size whose points fill their waves closely:
//   1-halo (5-D): 11 x 93 = 1023 points, 5 x 93 = 465 of 512, 2 x 93 = 186 of 192,
//                 4 x 93 = 372 of 384;
//   2-halo (6-D):  6 x 149 = 894 points of 896 (u_NFW pass 6 x 318 = 1908 in
//                  three rounds), 2 x 149 = 298 of 320, 1 x 149 of 192,
//                  3 x 149 = 447 of 512;
//   3-halo (7-D):  4 x 241 = 964 points, 2 x 241 = 482 of 512, 1 x 241 of 256,
//                  3 x 241 = 723 of 768.
template <int KV>
struct KGroup {
  static constexpr int D = kind_dim(kind_of_kv(KV));
  static constexpr int V = variant_of_kv(KV);
  static constexpr int P = rule_points(D);
  static constexpr int G = D == 5   ? (V == 3 ? 4 : V == 2 ? 2 : V ? 5 : 11)
                           : D == 6 ? (V == 3 ? 3 : V == 2 ? 1 : V ? 2 : 6)
                                    : (V == 3 ? 3 : V == 2 ? 1 : V ? 2 : 4);
  // the 2-halo kinds at three regions take 512 threads rather than 448, so
  // that their 954 u_NFW items fit two per thread
  static constexpr int NT = D == 6 && V == 3 ? 512 : (G * P + 63) / 64 * 64;
  static_assert(NT <= 1024, "one block holds every point of its regions");
};

// Region staging of the evaluation kernels: centre, half-width, volume, slot
// and integral parameters of the block's regions.
template <int D, int G>
struct Stage {
  double c[G][D];
  double h[G][D];
  double vol[G];
  uint32_t slot[G];
  TermArgs args[G];
};

// The group of G list entries (regions) this block evaluates.  A grid's
// blocks are dealt to the eight XCDs in turn (block b to XCD b mod 8), each
// XCD with its own L2, and neighbouring list entries mostly hold neighbouring
// slots of every geometry field; so each XCD takes runs of C consecutive
// groups (one run per XCD in turn) rather than every eighth group, and the
// runs stay short enough that every XCD still sees a mix of the list's
// integrals.  A bijection on [0, gridDim.x) whatever the dispatch order (the
// tail beyond the last full round of runs keeps its order): the results do
// not depend on it.
__device__ __forceinline__ uint32_t block_group() {
  constexpr uint32_t X = 8, C = 16;
  const uint32_t b = blockIdx.x, full = gridDim.x / (X * C) * (X * C);
  if (b >= full) return b;
  const uint32_t x = b % X, i = b / X;
  return ((i / C) * X + x) * C + i % C;
}

template <int D, int G, int NT>
__device__ __forceinline__ int stage_regions(const EvalLaunch &L, const EvalItem *list,
                                             uint32_t count, uint32_t group, Stage<D, G> &S) {
  const int tid = threadIdx.x;
  const uint32_t first = group * G;
  const int ng = (count - first) < (uint32_t)G ? (int)(count - first) : G;
  const uint64_t St = L.stride;
  if (tid < ng) {
    EvalItem it = list[first + tid];
    bool ok = it.slot < St && it.job < L.njobs;
    S.slot[tid] = ok ? it.slot : 0xffffffffu;
    if (ok) {
      S.args[tid] = L.args[L.jobs[it.job].args];
      S.vol[tid] = L.geo[kFieldVol * St + it.slot];
    }
  }
  __syncthreads();
  for (int i = tid; i < ng * D; i += NT) {
    int g = i / D, d = i - g * D;
    uint32_t sl = S.slot[g];
    if (sl == 0xffffffffu) continue;
    S.c[g][d] = L.geo[(kFieldC + d) * St + sl];
    S.h[g][d] = L.geo[(kFieldH + d) * St + sl];
  }
  __syncthreads();
  return ng;
}

// Rule reduction of the block's regions from the point values in f: lanes 2g
// and 2g + 1 of the first wave sum region g's 4th and 5th point groups
// (gm_group_sum), and lane 2g finishes the region.
template <int D, int G, int NP>
__device__ __forceinline__ void reduce_regions(const EvalLaunch &L, const Stage<D, G> &S,
                                               const double *f, int ng) {
  const int tid = threadIdx.x;
  const uint64_t St = L.stride;
  static_assert(2 * G <= 64, "a region's two lanes are in the first wave");
  if (tid < 2 * ng) {
    const int g = tid >> 1;
    const bool fifth = tid & 1;
    const double *v = f + g * NP;
    const double s = gm_group_sum<D>(v, fifth);
    const double s5 = __shfl_xor(s, 1);   // every lane below 2 ng is here
    if (!fifth && S.slot[g] != 0xffffffffu) {
      double val, err;
      int split = 0;
      gm_finish<D>(v, S.vol[g], s, s5, val, err, split);
      const uint32_t sl = S.slot[g];
      L.geo[kFieldVal * St + sl] = val;
      L.geo[kFieldErr * St + sl] = err;
      L.split[sl] = (uint8_t)split;
    }
  }
}

// ---------------------------------------------------- factored evaluation
// The NNMap/NMapMap integrands evaluated in three passes per block:
//   1. per region, each distinct value of the one- and two-coordinate
//      quantities: l1, l2 and their filters, cos phi, the redshift look-ups,
//      and per mass coordinate the mass, its indices, r_200 and the HOD
//      occupations (a function of (m, z));
//   2. per region, each distinct value of the u_NFW calls that depend on
//      part of the coordinates (33 of 93 points for u(k1, m, z) in 5-D) and
//      of the tree-level bispectrum (57 of 241 points in 7-D);
//   3. per point, the rest (u_NFW of k3 where it depends on every
//      coordinate, the products) from the cached values.
// Each cached value is computed by the same expressions from the same
// coordinates as in DirectSrc, so the point values are bit-identical.

// 72 bytes: it and zt (table indices below 2^16) share a word, so that a
// record's stride across the LDS banks stays 18 dwords.
struct MassC {
  double m, L, r200;
  int ir;
  uint16_t it, zt;
  double nc1, ns1, nc2, ns2, nss;
};
static_assert(sizeof(MassC) == 72, "MassC stride");

// u_NFW normalisation (c, ln(1+c), F) per f selector (1, f1, f2).
struct NfwC {
  double c[3], lc[3], F[3];
};

// Whether pass 1 caches the u_NFW normalisations per (mass, z) class (5-D and
// 6-D kinds).  The 7-D kinds compute them per u_NFW item: their classes are
// few, their pass 1 is the longest, and the larger cache costs them more than
// the logarithms it saves.
template <int KIND>
constexpr bool cache_nfw() { return Spec<kind_of_kv(KIND)>::D <= 6; }

// Whether pass 1 runs in two stages (the kinds that cache the NFW
// normalisations): the masses first, then the occupations and the
// normalisations as items of their own.  A (mass, z) item that does all of it
// is the pass's longest by far (pow, log, cbrt, two erf/exp occupations,
// three normalisations), and the block's other waves wait for it at the
// barrier; staged, the longest item is about a third as long, with one more
// barrier and no work repeated (NNMap 1h launches 3 %, 2h 1 % faster).
template <int KIND>
constexpr bool staged_p1() { return Spec<kind_of_kv(KIND)>::D <= 6; }

template <int KIND, int I>
struct UF {
  static constexpr int D = Spec<kind_of_kv(KIND)>::D;
  static constexpr USpec s = Spec<kind_of_kv(KIND)>::u[I];
  static constexpr int n = ProjTab<D, s.mask>::n;
};
// Offset of u factor I in the flat cache, in units of regions x classes.
template <int KIND, int I>
struct UOff {
  static constexpr int v = UOff<KIND, I - 1>::v + KGroup<KIND>::G * UF<KIND, I - 1>::n;
};
template <int KIND>
struct UOff<KIND, 0> {
  static constexpr int v = 0;
};

template <int KIND>
struct Cache {
  using S = Spec<kind_of_kv(KIND)>;
  static constexpr int D = S::D, G = KGroup<KIND>::G;
  static constexpr int NU_TOTAL = UOff<KIND, S::NU>::v;
  static constexpr int NB = S::has_bilin ? ProjTab<D, bilin_mask<D>()>::n : 1;
  static_assert(ProjTab<D, kL1>::n == 7 && ProjTab<D, kL2>::n == 7 &&
                    ProjTab<D, bit(2)>::n == 7 && ProjTab<D, bit(D - 1)>::n == 7,
                "seven coordinates per dimension");
  static_assert(ProjTab<D, kL1 | bit(D - 1)>::n == 17 && ProjTab<D, kL2 | bit(D - 1)>::n == 17,
                "seventeen (l, z) classes");
  static_assert(ProjTab<D, bit(S::mdim[0]) | bit(D - 1)>::n == 17 &&
                    ProjTab<D, bit(S::mdim[1]) | bit(D - 1)>::n == 17 &&
                    ProjTab<D, bit(S::mdim[2]) | bit(D - 1)>::n == 17,
                "seventeen (mass, z) classes");
  double l1[G][7], ap1[G][7], l2[G][7], ap2[G][7], cphi[G][7], z[G][7], w[G][7];
  double zpre[G][7], zfac[G][7];
  double rw[G][7];   // 1/w, correctly rounded: k = l / w by div_rn
  // NNMap 3-halo: dwdz, 1/dwdz, g, p1, p2, 1/w per redshift (proj_3h)
  double ztab[kind_of_kv(KIND) == kNN3 ? G : 1][7][6];
  int zr[G][7], zt[G][7];
  MassC m[S::NM][G][17];
  NfwC nf[cache_nfw<KIND>() ? S::NM : 1][cache_nfw<KIND>() ? G : 1][17];
  double pk[S::has_pk ? 2 : 1][G][17];  // P(k1), P(k2) per (l, z) class
  static constexpr int N3 = ProjTab<D, kL3>::n;             // (l1, l2, phi) classes
  static constexpr int N3Z = ProjTab<D, kL3 | bit(D - 1)>::n;  // (l1, l2, phi, z) classes
  double l3[G][N3], ap3[G][N3];
  double pk3[S::has_pk ? G : 1][N3Z];                      // P(k3), 2-halo terms
  double u[NU_TOTAL];
  double bl[G * NB];
};

// Class indices of every point in one 16-byte load; a byte load with its address
// arithmetic per index, and whole rule points rebuilt for one or two of their
// coordinates, were a good part of a point's instructions.  Packed look-ups, coordinates
// by code and quotients by known reciprocals (DevTables) together took the
// evaluation of the 550-triplet workload from 281 to 254 ms, values
// bit-identical.  Word 0 l1, l2, z (3 bits each), l3 (6),
// the masses' (5 each); word 1 (l1, z), (l2, z) (5 each), (l1, l2, phi, z) (7)
// and u factors 0 and 1 (7 each); word 2 u factors 2 to 5 (7 each).
struct PointWords {
  uint32_t w0, w1, w2, pad;
};
template <int KIND>
constexpr Packed<rule_points(Spec<kind_of_kv(KIND)>::D), PointWords> make_points() {
  using S = Spec<kind_of_kv(KIND)>;
  constexpr int D = S::D;
  constexpr unsigned z = bit(D - 1);
  constexpr auto l1 = make_proj<D, kL1>();
  constexpr auto l2 = make_proj<D, kL2>();
  constexpr auto pz = make_proj<D, z>();
  constexpr auto l3 = make_proj<D, kL3>();
  constexpr auto m0 = make_proj<D, bit(S::mdim[0]) | z>();
  constexpr auto m1 = make_proj<D, bit(S::mdim[S::NM > 1 ? 1 : 0]) | z>();
  constexpr auto m2 = make_proj<D, bit(S::mdim[S::NM > 2 ? 2 : 0]) | z>();
  constexpr auto l1z = make_proj<D, kL1 | z>();
  constexpr auto l2z = make_proj<D, kL2 | z>();
  constexpr auto l3z = make_proj<D, kL3 | z>();
  constexpr auto u0 = make_proj<D, S::u[0].mask>();
  constexpr auto u1 = make_proj<D, S::u[1].mask>();
  constexpr auto u2 = make_proj<D, S::u[2].mask>();
  constexpr auto u3 = make_proj<D, S::u[S::NU > 3 ? 3 : 0].mask>();
  constexpr auto u4 = make_proj<D, S::u[S::NU > 4 ? 4 : 0].mask>();
  constexpr auto u5 = make_proj<D, S::u[S::NU > 5 ? 5 : 0].mask>();
  static_assert(l3.n <= 64 && l3z.n <= 128 && u0.n <= 128 && u1.n <= 128 && u2.n <= 128 &&
                u3.n <= 128 && u4.n <= 128 && u5.n <= 128 && m0.n <= 32, "field widths");
  Packed<rule_points(D), PointWords> t{};
  for (int q = 0; q < rule_points(D); ++q) {
    t.w[q].w0 = l1.cls[q] | l2.cls[q] << 3 | pz.cls[q] << 6 | l3.cls[q] << 9 | m0.cls[q] << 15 |
                m1.cls[q] << 20 | (uint32_t)m2.cls[q] << 25;
    t.w[q].w1 = l1z.cls[q] | l2z.cls[q] << 5 | l3z.cls[q] << 10 | u0.cls[q] << 17 |
                (uint32_t)u1.cls[q] << 24;
    t.w[q].w2 = u2.cls[q] | u3.cls[q] << 7 | u4.cls[q] << 14 | (uint32_t)u5.cls[q] << 21;
  }
  return t;
}
template <int KIND>
__constant__ constexpr auto kPoints = make_points<kind_of_kv(KIND)>();

// Per class of a u factor: its l (6 bits), z (3) and mass (5) classes.
template <int KIND, int I>
constexpr auto make_u_words() {
  using S = Spec<KIND>;
  constexpr int D = S::D;
  constexpr USpec s = S::u[I];
  constexpr auto p = make_proj<D, s.mask>();
  constexpr auto l = make_proj<D, s.kidx == 1 ? kL1 : s.kidx == 2 ? kL2 : kL3>();
  constexpr auto pz = make_proj<D, bit(D - 1)>();
  constexpr auto pm = make_proj<D, bit(S::mdim[s.slot]) | bit(D - 1)>();
  Packed<p.n> t{};
  for (int c = 0; c < p.n; ++c)
    t.w[c] = (uint16_t)(l.cls[p.rep[c]] | pz.cls[p.rep[c]] << 6 | pm.cls[p.rep[c]] << 9);
  return t;
}
template <int KIND, int I>
__constant__ constexpr auto kUWords = make_u_words<KIND, I>();

// Per (l1, l2, phi) or (l1, l2, phi, z) class: the classes of l1, l2, phi, z
// (3 bits each), and for the latter of l3 (6 bits).
template <int D, unsigned MASK>
constexpr auto make_geo_words() {
  constexpr auto p = make_proj<D, MASK>();
  constexpr auto l1 = make_proj<D, kL1>();
  constexpr auto l2 = make_proj<D, kL2>();
  constexpr auto ph = make_proj<D, bit(2)>();
  constexpr auto pz = make_proj<D, bit(D - 1)>();
  constexpr auto l3 = make_proj<D, kL3>();
  Packed<p.n, uint32_t> t{};
  for (int c = 0; c < p.n; ++c) {
    const int q = p.rep[c];
    t.w[c] = l1.cls[q] | l2.cls[q] << 3 | ph.cls[q] << 6 | pz.cls[q] << 9 | l3.cls[q] << 12;
  }
  return t;
}
template <int D, unsigned MASK>
__constant__ constexpr auto kGeoWords = make_geo_words<D, MASK>();
// Codes of the (mass, z) classes by mass slot, and of the (l1, z), (l2, z) ones.
template <int KIND>
__constant__ constexpr auto kMassCodes =
    make_codes<Spec<KIND>::D, Spec<KIND>::mdim[0], Spec<KIND>::mdim[Spec<KIND>::NM > 1 ? 1 : 0],
               Spec<KIND>::mdim[Spec<KIND>::NM > 2 ? 2 : 0]>();
template <int D>
__constant__ constexpr auto kLCodes = make_codes<D, 0, 1, 1>();
__device__ __forceinline__ uint32_t bits(uint32_t w, int at, int n) {
  return (w >> at) & ((1u << n) - 1u);
}

// Per-point view of the cache (the value source of the integrands).
template <int KIND, class P>
struct CachedSrc {
  using S = Spec<kind_of_kv(KIND)>;
  static constexpr int D = S::D, G = KGroup<KIND>::G;
  const Cache<KIND> &C;
  const TermArgs &a;
  int g;
  PointWords pw;
  Geo G_;
  __device__ __forceinline__ CachedSrc(const Cache<KIND> &C_, const TermArgs &a_, int g_, int q)
      : C(C_), a(a_), g(g_), pw(kPoints<kind_of_kv(KIND)>.w[q]) {
    G_ = Geo{};
    G_.l1 = C.l1[g][c1()];
    G_.l2 = C.l2[g][c2()];
    G_.zr = C.zr[g][cz()];
  }
  __device__ __forceinline__ uint32_t c1() const { return bits(pw.w0, 0, 3); }
  __device__ __forceinline__ uint32_t c2() const { return bits(pw.w0, 3, 3); }
  __device__ __forceinline__ uint32_t cz() const { return bits(pw.w0, 6, 3); }
  __device__ __forceinline__ const MassC &mc(int i) const {
    if (i == 0) return C.m[0][g][bits(pw.w0, 15, 5)];
    if (S::NM > 1 && i == 1) return C.m[S::NM > 1 ? 1 : 0][g][bits(pw.w0, 20, 5)];
    return C.m[S::NM > 2 ? 2 : 0][g][bits(pw.w0, 25, 5)];
  }
  __device__ __forceinline__ const Geo &geo() const { return G_; }
  __device__ __forceinline__ Mass mass(int i) const {
    const MassC &e = mc(i);
    Mass M;
    M.m = e.m;
    M.L = e.L;
    M.ir = e.ir;
    M.it = e.it;
    M.r200 = e.r200;
    return M;
  }
  __device__ __forceinline__ Occ occ1(int i) const {
    const MassC &e = mc(i);
    return Occ{e.nc1, e.ns1};
  }
  __device__ __forceinline__ Occ occ2(int i) const {
    const MassC &e = mc(i);
    return Occ{e.nc2, e.ns2};
  }
  __device__ __forceinline__ double nss(int i) const { return mc(i).nss; }
  template <int I>
  __device__ __forceinline__ double u() const {
    using F = UF<KIND, I>;
    const uint32_t c = I == 0   ? bits(pw.w1, 17, 7)
                       : I == 1 ? bits(pw.w1, 24, 7)
                                : bits(pw.w2, I < 2 ? 0 : 7 * (I - 2), 7);
    return C.u[UOff<KIND, I>::v + g * F::n + c];
  }
  __device__ __forceinline__ double ap1() const { return C.ap1[g][c1()]; }
  __device__ __forceinline__ double ap2() const { return C.ap2[g][c2()]; }
  __device__ __forceinline__ double bl() const {
    return C.bl[g * Cache<KIND>::NB + bits(pw.w1, 10, 7)];
  }
  __device__ __forceinline__ double ap3() const { return C.ap3[g][bits(pw.w0, 9, 6)]; }
  __device__ __forceinline__ double pk3() const {
    return C.pk3[S::has_pk ? g : 0][bits(pw.w1, 10, 7)];
  }
  __device__ __forceinline__ double pk1() const { return C.pk[0][g][bits(pw.w1, 0, 5)]; }
  __device__ __forceinline__ double pk2() const {
    return C.pk[S::has_pk ? 1 : 0][g][bits(pw.w1, 5, 5)];
  }
  __device__ __forceinline__ double zpre() const { return C.zpre[g][cz()]; }
  __device__ __forceinline__ double proj(double B) const {
    if constexpr (kind_of_kv(KIND) == kNN3) {
      const double *t = C.ztab[g][cz()];
      return proj_3h(B, t[0], t[1], t[2], t[3], t[4], C.w[g][cz()], t[5], C.z[g][cz()]);
    } else {
      return C.zfac[g][cz()] * B;
    }
  }
};

// Pass 1 item layout: wave-aligned segments of items that run the same code:
// l1 and l2 with their filters (2 x G x 7), cos phi (G x 7), the redshift
// look-ups and z-only factors (G x 7), every mass coordinate's (m, z) class
// (NM x G x 17; the coordinates of one kind need the same u_NFW
// normalisations), and for the 2-halo terms P(k1), P(k2) per (l, z) class
// (2 x G x 17).
template <int KIND>
struct P1Layout {
  using S = Spec<kind_of_kv(KIND)>;
  static constexpr int G = KGroup<KIND>::G;
  static constexpr int pad(int n) { return (n + 63) / 64 * 64; }
  static constexpr int L = 0, PHI = pad(2 * G * 7), Z = PHI + pad(G * 7), MZ = Z + pad(G * 7);
  static constexpr int PK = MZ + pad(S::NM * G * 17);
  static constexpr int END = PK + (S::has_pk ? pad(2 * G * 17) : 0);
};

template <int KIND, class P>
__device__ __forceinline__ void pass1(const DevTables &T, const Stage<Spec<kind_of_kv(KIND)>::D, KGroup<KIND>::G> &St,
                                      Cache<KIND> &C, int i, int ng) {
  using S = Spec<kind_of_kv(KIND)>;
  using Lay = P1Layout<KIND>;
  constexpr int D = S::D, G = KGroup<KIND>::G;
  static_assert(single_codes<D, 0>() && single_codes<D, 1>() && single_codes<D, 2>() &&
                    single_codes<D, D - 1>(), "coordinate codes by class");
  if (i < Lay::PHI) {
    const int r = i - Lay::L;
    if (r >= 2 * G * 7) return;
    const int which = r / (G * 7), rr = r - which * G * 7, g = rr / 7, c = rr - g * 7;
    if (g >= ng || St.slot[g] == 0xffffffffu) return;
    const TermArgs &a = St.args[g];
    // l1 and l2 items share one wave: one code path with selected operands
    const double l = P::l(rule_coord(single_code(c), St.c[g][which], St.h[g][which]));
    const double ap = P::ap((which == 0 ? a.t1 : a.t2) * l);
    if (which == 0) {
      C.l1[g][c] = l;
      C.ap1[g][c] = ap;
    } else {
      C.l2[g][c] = l;
      C.ap2[g][c] = ap;
    }
  } else if (i < Lay::Z) {
    const int r = i - Lay::PHI;
    if (r >= G * 7) return;
    const int g = r / 7, c = r - g * 7;
    if (g >= ng || St.slot[g] == 0xffffffffu) return;
    C.cphi[g][c] = cos(rule_coord(single_code(c), St.c[g][2], St.h[g][2]));
  } else if (i < Lay::MZ) {
    const int r = i - Lay::Z;
    if (r >= G * 7) return;
    const int g = r / 7, c = r - g * 7;
    if (g >= ng || St.slot[g] == 0xffffffffu) return;
    const double z = rule_coord(single_code(c), St.c[g][D - 1], St.h[g][D - 1]);
    const int zr = zix_round(T, z);
    const double w = T.w[zr];
    C.z[g][c] = z;
    C.zr[g][c] = zr;
    C.zt[g][c] = zix_trunc(T, z);
    C.w[g][c] = w;
    C.rw[g][c] = T.rw[zr];
    zfactors<kind_of_kv(KIND)>(T, St.args[g], zr, z, w, C.zpre[g][c], C.zfac[g][c]);
    if constexpr (kind_of_kv(KIND) == kNN3) {
      double *t = C.ztab[g][c];
      t[0] = T.dwdz[zr];
      t[1] = 1. / t[0];
      t[2] = T.g[zr];
      t[3] = T.p1[zr];
      t[4] = T.p2[zr];
      t[5] = T.rw[zr];
    }
  } else if (i < Lay::PK) {
    const int r = i - Lay::MZ;
    if (r >= S::NM * G * 17) return;
    const int slot = r / (G * 17), rr = r - slot * G * 17, g = rr / 17, c = rr - g * 17;
    if (g >= ng || St.slot[g] == 0xffffffffu) return;
    const TermArgs &a = St.args[g];
    const int md = slot == 0 ? S::mdim[0] : slot == 1 ? S::mdim[1] : S::mdim[2];
    const uint32_t code = kMassCodes<kind_of_kv(KIND)>.w[slot * 17 + c];
    const int zt = zix_trunc(T, rule_coord(code >> 4, St.c[g][D - 1], St.h[g][D - 1]));
    const Mass M = make_mass<P>(T, rule_coord(code & 7, St.c[g][md], St.h[g][md]), zt);
    MassC &e = C.m[slot][g][c];
    e.m = M.m;
    e.L = M.L;
    e.r200 = M.r200;
    e.ir = M.ir;
    e.it = (uint16_t)M.it;
    e.zt = (uint16_t)zt;
    if constexpr (staged_p1<KIND>()) return;   // the rest in pass1b
    if constexpr (kind_of_kv(KIND) == kNN3) {
      // the NNMap 3-halo term needs the first HOD at m1 and the second at m2
      // only: one occupation per item, the HOD selected by the mass slot
      const bool second = slot == 1;
      const Occ o = P::occ(second ? a.h2 : a.h1, second ? a.rs2 : a.rs1,
                           second ? a.lth2 : a.lth1, second ? a.lmp2 : a.lmp1, M);
      e.nc1 = e.nc2 = o.nc;
      e.ns1 = e.ns2 = o.ns;
    } else {
      const Occ o1 = occ1<P>(a, M);
      e.nc1 = o1.nc;
      e.ns1 = o1.ns;
      if constexpr (S::two_hods) {
        const Occ o2 = occ2<P>(a, M);
        e.nc2 = o2.nc;
        e.ns2 = o2.ns;
        if (slot == S::nss_slot) e.nss = nsatnsat<P>(a, o1.ns, o2.ns, M);
      }
    }
    if constexpr (cache_nfw<KIND>()) {
      NfwC &en = C.nf[slot][g][c];
#pragma unroll
      for (int fs = 0; fs < 3; ++fs) {
        const bool need = slot == 0 ? uses_nfw<kind_of_kv(KIND)>(0, fs)
                                    : slot == 1 ? uses_nfw<kind_of_kv(KIND)>(1, fs) : uses_nfw<kind_of_kv(KIND)>(2, fs);
        if (need) {
          const Nfw nf = make_nfw<P>(T, M, zt, f_of(a, fs));
          en.c[fs] = nf.c;
          en.lc[fs] = nf.lc;
          en.F[fs] = nf.F;
        }
      }
    }
  } else if constexpr (S::has_pk) {
    const int r = i - Lay::PK;
    if (r >= 2 * G * 17) return;
    const int which = r / (G * 17), rr = r - which * G * 17, g = rr / 17, c = rr - g * 17;
    if (g >= ng || St.slot[g] == 0xffffffffu) return;
    // P(k) at k = l / w, the same expressions as the per-point Geo
    const uint32_t code = kLCodes<D>.w[which * 17 + c];
    const double l = P::l(rule_coord(code & 7, St.c[g][which], St.h[g][which]));
    const int zr = zix_round(T, rule_coord(code >> 4, St.c[g][D - 1], St.h[g][D - 1]));
    C.pk[which][g][c] = pk(T, zr, div_rn(l, T.w[zr], T.rw[zr]));
  }
}

// Second stage of pass 1 (staged_p1 kinds): item i is one of a (mass, z)
// class's NFW normalisations (3 x NM x G x 17 items, one per f selector) or
// HOD occupations (the first HOD's, and the second's for the two-HOD kinds:
// NM x G x 17 items each), from the masses of the first stage, or l3 with its
// aperture filter per (l1, l2, phi) class (G x N3 items), from the first
// stage's l1, l2 and cos phi.  NsatNsat, which needs both occupations, is a
// pass-2 item.  The normalisations come first: where a thread takes a second
// item, its first is one of the shortest.
template <int KIND>
struct P1bLayout {
  using S = Spec<kind_of_kv(KIND)>;
  static constexpr int G = KGroup<KIND>::G;
  static constexpr int pad(int n) { return (n + 63) / 64 * 64; }
  static constexpr int NMZ = S::NM * G * 17;
  static constexpr int OCC1 = pad(3 * NMZ), OCC2 = OCC1 + pad(NMZ);
  static constexpr int L3 = OCC2 + (S::two_hods ? pad(NMZ) : 0);
  static constexpr int END = L3 + pad(G * ProjTab<S::D, kL3>::n);
};

__device__ __forceinline__ Mass mass_of(const MassC &e) {
  Mass M;
  M.m = e.m;
  M.L = e.L;
  M.ir = e.ir;
  M.it = e.it;
  M.r200 = e.r200;
  return M;
}

template <int KIND, class P>
__device__ __forceinline__ void pass1b(const DevTables &T, const Stage<Spec<kind_of_kv(KIND)>::D, KGroup<KIND>::G> &St,
                                       Cache<KIND> &C, int i, int ng) {
  using S = Spec<kind_of_kv(KIND)>;
  using Lay = P1bLayout<KIND>;
  constexpr int D = S::D, G = KGroup<KIND>::G;
  if (i < Lay::OCC1) {
    if (i >= 3 * Lay::NMZ) return;
    const int fs = i / Lay::NMZ, rm = i - fs * Lay::NMZ;
    const int slot = rm / (G * 17), rr = rm - slot * G * 17, g = rr / 17, c = rr - g * 17;
    const bool need = slot == 0 ? uses_nfw<kind_of_kv(KIND)>(0, fs)
                                : slot == 1 ? uses_nfw<kind_of_kv(KIND)>(1, fs) : uses_nfw<kind_of_kv(KIND)>(2, fs);
    if (!need || g >= ng || St.slot[g] == 0xffffffffu) return;
    const MassC &e = C.m[slot][g][c];
    const Nfw nf = make_nfw<P>(T, mass_of(e), e.zt, f_of(St.args[g], fs));
    NfwC &en = C.nf[slot][g][c];
    en.c[fs] = nf.c;
    en.lc[fs] = nf.lc;
    en.F[fs] = nf.F;
    return;
  }
  if (i < Lay::L3) {
    const bool second = i >= Lay::OCC2;
    const int r = i - (second ? Lay::OCC2 : Lay::OCC1);
    if (r >= Lay::NMZ) return;
    const int slot = r / (G * 17), rr = r - slot * G * 17, g = rr / 17, c = rr - g * 17;
    if (g >= ng || St.slot[g] == 0xffffffffu) return;
    MassC &e = C.m[slot][g][c];
    const Mass M = mass_of(e);
    const TermArgs &a = St.args[g];
    if (!second) {
      const Occ o = occ1<P>(a, M);
      e.nc1 = o.nc;
      e.ns1 = o.ns;
    } else if constexpr (S::two_hods) {
      const Occ o = occ2<P>(a, M);
      e.nc2 = o.nc;
      e.ns2 = o.ns;
    }
    return;
  }
  // l3 and its filter per (l1, l2, phi) class, the expressions of the Geo
  constexpr int N3 = Cache<KIND>::N3;
  const int r = i - Lay::L3;
  if (r >= G * N3) return;
  const int g = r / N3, c = r - g * N3;
  if (g >= ng || St.slot[g] == 0xffffffffu) return;
  const uint32_t gw = kGeoWords<D, kL3>.w[c];
  const double l1 = C.l1[g][bits(gw, 0, 3)], l2 = C.l2[g][bits(gw, 3, 3)];
  const double l3 = sqrt(l1 * l1 + l2 * l2 + 2 * l1 * l2 * C.cphi[g][bits(gw, 6, 3)]);
  C.l3[g][c] = l3;
  C.ap3[g][c] = P::ap(St.args[g].t3 * l3);
}

// Pass 2: the inputs of u-factor item i (factor I or later).
template <int KIND, class P, int I>
__device__ __forceinline__ bool u_inputs(const DevTables &T,
                                         const Stage<Spec<kind_of_kv(KIND)>::D, KGroup<KIND>::G> &St,
                                         const Cache<KIND> &C, int i, int ng, int &dst, Nfw &n,
                                         double &k, uint32_t &nfe) {
  using S = Spec<kind_of_kv(KIND)>;
  if constexpr (I >= S::NU) {
    return false;
  } else {
    constexpr int D = S::D;
    using F = UF<KIND, I>;
    constexpr int lo = UOff<KIND, I>::v, hi = UOff<KIND, I + 1>::v;
    if (i >= hi) return u_inputs<KIND, P, I + 1>(T, St, C, i, ng, dst, n, k, nfe);
    const int r = i - lo, g = r / F::n, c = r - g * F::n;
    if (g >= ng || St.slot[g] == 0xffffffffu) return false;
    const uint32_t uw = kUWords<kind_of_kv(KIND), I>.w[c];
    const uint32_t cl = bits(uw, 0, 6), cz = bits(uw, 6, 3), cm = bits(uw, 9, 5);
    const double w = C.w[g][cz];
    double l;
    if constexpr (F::s.kidx == 1) {
      l = C.l1[g][cl];
    } else if constexpr (F::s.kidx == 2) {
      l = C.l2[g][cl];
    } else if constexpr (staged_p1<KIND>()) {
      l = C.l3[g][cl];   // from pass 1, the same expression
    } else {
      const uint32_t gw = kGeoWords<D, kL3>.w[cl];
      const double l1 = C.l1[g][bits(gw, 0, 3)], l2 = C.l2[g][bits(gw, 3, 3)];
      l = sqrt(l1 * l1 + l2 * l2 + 2 * l1 * l2 * C.cphi[g][bits(gw, 6, 3)]);
    }
    k = div_rn(l, w, C.rw[g][cz]);   // = l / w (IEEE), in three instructions
    const MassC &e = C.m[F::s.slot][g][cm];
    if constexpr (cache_nfw<KIND>()) {
      const NfwC &en = C.nf[F::s.slot][g][cm];
      n = Nfw{e.r200, en.c[F::s.fsel], en.lc[F::s.fsel], en.F[F::s.fsel]};
      // the normalisations' entry in C.nf (flat), times 4, plus the f selector
      nfe = (uint32_t)(((F::s.slot * KGroup<KIND>::G + g) * 17 + cm) * 4 + F::s.fsel);
    } else {
      Mass M;
      M.m = e.m;
      M.L = e.L;
      M.ir = e.ir;
      M.it = e.it;
      M.r200 = e.r200;
      n = make_nfw<P>(T, M, C.zt[g][cz], f_of(St.args[g], F::s.fsel));
    }
    dst = i;
    return true;
  }
}

// Pass 2 item layout: the u_NFW items, then (64-aligned) the bispectrum
// items, l3 with its filter per (l1, l2, phi) class, and for the 2-halo terms
// P(k3) per (l1, l2, phi, z) class.
template <int KIND>
struct P2Layout {
  using S = Spec<kind_of_kv(KIND)>;
  static constexpr int G = KGroup<KIND>::G;
  static constexpr int pad(int n) { return (n + 63) / 64 * 64; }
  static constexpr int UPAD = pad(Cache<KIND>::NU_TOTAL);
  static constexpr int L3 = UPAD + (S::has_bilin ? pad(G * Cache<KIND>::NB) : 0);
  static constexpr int PK3 = L3 + (staged_p1<KIND>() ? 0 : pad(G * Cache<KIND>::N3));
  // NsatNsat per (mass, z) class of its mass coordinate, where pass 1 runs
  // in two stages (the occupations are then separate items)
  static constexpr int NSS = PK3 + (S::has_pk ? pad(G * Cache<KIND>::N3Z) : 0);
  static constexpr bool kNss = staged_p1<KIND>() && S::two_hods && S::nss_slot >= 0;
  static constexpr int END = NSS + (kNss ? pad(G * 17) : 0);
};

// Pass 2 items after the u_NFW ones (i >= the u items' padded count).
template <int KIND, class P>
__device__ __forceinline__ void pass2_rest(const DevTables &T, const Stage<Spec<kind_of_kv(KIND)>::D, KGroup<KIND>::G> &St,
                                           Cache<KIND> &C, int i, int ng) {
  using S = Spec<kind_of_kv(KIND)>;
  constexpr int D = S::D, G = KGroup<KIND>::G;
  constexpr int NU_TOTAL = Cache<KIND>::NU_TOTAL;
  constexpr int UPAD = (NU_TOTAL + 63) / 64 * 64;
  using Lay = P2Layout<KIND>;
  if constexpr (Lay::kNss) {
    if (i >= Lay::NSS) {
      const int r = i - Lay::NSS;
      if (r >= G * 17) return;
      const int g = r / 17, c = r - g * 17;
      if (g >= ng || St.slot[g] == 0xffffffffu) return;
      MassC &e = C.m[S::nss_slot > 0 ? S::nss_slot : 0][g][c];
      e.nss = nsatnsat<P>(St.args[g], e.ns1, e.ns2, mass_of(e));
      return;
    }
  }
  if (i < Lay::L3) {
    if constexpr (S::has_bilin) {
      constexpr int NB = Cache<KIND>::NB;
      const int r = i - UPAD;
      if (r < 0 || r >= G * NB) return;
      const int g = r / NB, c = r - g * NB;
      if (g >= ng || St.slot[g] == 0xffffffffu) return;
      const uint32_t gw = kGeoWords<D, bilin_mask<D>()>.w[c];
      const uint32_t cz = bits(gw, 9, 3);
      const double w = C.w[g][cz], rw = C.rw[g][cz];
      const double k1 = div_rn(C.l1[g][bits(gw, 0, 3)], w, rw);
      const double k2 = div_rn(C.l2[g][bits(gw, 3, 3)], w, rw);
      C.bl[r] = bilin(T, k1, k2, C.cphi[g][bits(gw, 6, 3)], C.z[g][cz]);
    }
    return;
  }
  if (i < Lay::PK3) {
    // l3 and its filter per (l1, l2, phi) class, the expressions of the Geo
    constexpr int N3 = Cache<KIND>::N3;
    const int r = i - Lay::L3;
    if (r >= G * N3) return;
    const int g = r / N3, c = r - g * N3;
    if (g >= ng || St.slot[g] == 0xffffffffu) return;
    const uint32_t gw = kGeoWords<D, kL3>.w[c];
    const double l1 = C.l1[g][bits(gw, 0, 3)], l2 = C.l2[g][bits(gw, 3, 3)];
    const double l3 = sqrt(l1 * l1 + l2 * l2 + 2 * l1 * l2 * C.cphi[g][bits(gw, 6, 3)]);
    C.l3[g][c] = l3;
    C.ap3[g][c] = P::ap(St.args[g].t3 * l3);
    return;
  }
  if constexpr (S::has_pk) {
    // P(k3) per (l1, l2, phi, z) class
    constexpr int N3Z = Cache<KIND>::N3Z;
    const int r = i - Lay::PK3;
    if (r >= G * N3Z) return;
    const int g = r / N3Z, c = r - g * N3Z;
    if (g >= ng || St.slot[g] == 0xffffffffu) return;
    const uint32_t gw = kGeoWords<D, kL3 | bit(D - 1)>.w[c];
    const uint32_t cz = bits(gw, 9, 3);
    double l3;
    if constexpr (staged_p1<KIND>()) {
      l3 = C.l3[g][bits(gw, 12, 6)];
    } else {
      const double l1 = C.l1[g][bits(gw, 0, 3)], l2 = C.l2[g][bits(gw, 3, 3)];
      l3 = sqrt(l1 * l1 + l2 * l2 + 2 * l1 * l2 * C.cphi[g][bits(gw, 6, 3)]);
    }
    C.pk3[g][c] = pk(T, C.zr[g][cz], div_rn(l3, C.w[g][cz], C.rw[g][cz]));
  }
}

template <int KIND, class P>
__device__ __forceinline__ void pass2(const DevTables &T, const Stage<Spec<kind_of_kv(KIND)>::D, KGroup<KIND>::G> &St,
                                      Cache<KIND> &C, int i, int ng) {
  if (i < Cache<KIND>::NU_TOTAL) {
    int dst;
    Nfw n;
    double k;
    uint32_t nfe;
    if (!u_inputs<KIND, P, 0>(T, St, C, i, ng, dst, n, k, nfe)) return;
    C.u[dst] = P::u(n, k);
    return;
  }
  pass2_rest<KIND, P>(T, St, C, i, ng);
}

// u_NFW items in branch order.  u_NFW has three branches (a1 >= 4,
// a1 < 4 <= a2, a2 < 4) and a wave runs every branch one of its lanes takes:
// on the 550-triplet workload about half of the waves of u items mix two or
// three branches and run about a third more instructions than their lanes
// need.  For the kinds that cache the NFW normalisations, pass 2 therefore (1) computes each u item's a1, keeps it
// in the item's own output slot and appends the item to its branch's list
// (one LDS atomic per wave), and (2) evaluates the items from the lists in
// branch order, so that a wave's lanes mostly share one branch.  Every item runs the same expressions on
// the same inputs either way: the values are bit-identical.
template <int KIND>
constexpr bool sort_u() { return cache_nfw<KIND>(); }

// Step 1 for u item i: a1 into C.u[i], its normalisations' entry into
// unf[i], and i into its branch's list: a1 >= 4 from the front of `ends`,
// a2 < 4 from the back of `ends`, a1 < 4 <= a2 from the front of `mid`.  The
// three branch counts of a wave are added to the block's counters (21-bit
// fields of one 64-bit word) by a single LDS atomic, whose old value gives
// each branch's base.
template <int KIND, class P>
__device__ __forceinline__ void u_classify(const DevTables &T,
                                           const Stage<Spec<kind_of_kv(KIND)>::D, KGroup<KIND>::G> &St,
                                           Cache<KIND> &C, int i, int ng, unsigned long long *cnt,
                                           uint16_t *unf, uint16_t *ends, uint16_t *mid) {
  constexpr int NU = Cache<KIND>::NU_TOTAL;
  int dst = 0;
  Nfw n;
  double k = 0;
  uint32_t nfe = 0;
  const bool ok = u_inputs<KIND, P, 0>(T, St, C, i, ng, dst, n, k, nfe);
  int b = 3;
  if (ok) {
    const double a1 = nfw_a1(n, k);
    C.u[dst] = a1;
    unf[dst] = (uint16_t)nfe;
    b = a1 >= 4 ? 0 : (a1 * (1 + n.c) >= 4 ? 1 : 2);
  }
  const uint64_t m0 = __ballot(b == 0), m1 = __ballot(b == 1), m2 = __ballot(b == 2);
  const uint64_t add = (uint64_t)__popcll(m0) | ((uint64_t)__popcll(m1) << 21) |
                       ((uint64_t)__popcll(m2) << 42);
  const int first = __ffsll((unsigned long long)__ballot(1)) - 1;
  uint64_t old = 0;
  if ((int)__lane_id() == first) old = atomicAdd(cnt, (unsigned long long)add);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)old, first);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(old >> 32), first);
  if (b == 3) return;
  const uint64_t o = ((uint64_t)hi << 32) | lo;
  const uint32_t base = (uint32_t)(o >> (21 * b)) & 0x1fffffu;
  const uint64_t m = b == 0 ? m0 : b == 1 ? m1 : m2;
  const uint32_t pos = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  if (b == 1) mid[pos] = (uint16_t)dst;
  else ends[b == 0 ? pos : NU - 1 - pos] = (uint16_t)dst;
}

// Step 1, round r of R over the pass-2 items tid + r NT: each round holds
// only the code its items can reach (u items, the rest, or both).
template <int KIND, class P, int r, int R>
__device__ __forceinline__ void sort_round(const DevTables &T,
                                           const Stage<Spec<kind_of_kv(KIND)>::D, KGroup<KIND>::G> &St,
                                           Cache<KIND> &C, int tid, int ng, unsigned long long *cnt,
                                           uint16_t *unf, uint16_t *ends, uint16_t *mid) {
  if constexpr (r < R) {
    constexpr int NT = KGroup<KIND>::NT, NU = Cache<KIND>::NU_TOTAL, P2 = P2Layout<KIND>::END;
    const int i = tid + r * NT;
    if constexpr ((r + 1) * NT <= NU) {
      u_classify<KIND, P>(T, St, C, i, ng, cnt, unf, ends, mid);
    } else if constexpr (r * NT >= NU) {
      if (i < P2) pass2_rest<KIND, P>(T, St, C, i, ng);
    } else {
      if (i < NU) u_classify<KIND, P>(T, St, C, i, ng, cnt, unf, ends, mid);
      else if (i < P2) pass2_rest<KIND, P>(T, St, C, i, ng);
    }
    sort_round<KIND, P, r + 1, R>(T, St, C, tid, ng, cnt, unf, ends, mid);
  }
}

// Step 3 for u item i, whose a1 is in C.u[i] and normalisations' entry in
// unf[i].
template <int KIND, class P>
__device__ __forceinline__ void u_eval_sorted(Cache<KIND> &C, int i, const uint16_t *unf) {
  const uint32_t e = unf[i];
  const NfwC &en = (&C.nf[0][0][0])[e >> 2];
  const int fs = e & 3;
  C.u[i] = P::u_a1(C.u[i], Nfw{0.0, en.c[fs], en.lc[fs], en.F[fs]});
}

// LDS of an evaluation block.
template <int KIND>
struct EvalLds {
  using S = Spec<kind_of_kv(KIND)>;
  static constexpr int G = KGroup<KIND>::G, NP = KGroup<KIND>::P;
  static constexpr int NU = Cache<KIND>::NU_TOTAL;
  static constexpr bool kSort = sort_u<KIND>();
  // f holds the point values of pass 3, and before that the branch lists of the
  // u items (2 NU entries of 16 bits)
  static constexpr int NF = kSort && (4 * NU + 7) / 8 > G * NP ? (4 * NU + 7) / 8 : G * NP;
  static constexpr int NUNF = kSort ? NU : 1;
  using Stg = Stage<S::D, G>;
  Stg St;
  Cache<KIND> C;
  double f[NF];
  unsigned long long ucnt;   // u items per branch, 21-bit fields
  uint16_t unf[NUNF];
};

// Evaluates group `group` of the list: its regions' values, errors and split
// dimensions.  The block has KGroup<KIND>::NT threads and all of them call it.
template <int KIND, class P>
__device__ __forceinline__ void eval_block(const EvalLaunch &L, const EvalItem *list,
                                           uint32_t count, uint32_t group,
                                           typename EvalLds<KIND>::Stg &St, Cache<KIND> &C,
                                           double *s_f, unsigned long long &s_ucnt,
                                           uint16_t *s_unf) {
  using S = Spec<kind_of_kv(KIND)>;
  constexpr int D = S::D;
  constexpr int NP = KGroup<KIND>::P;
  constexpr int G = KGroup<KIND>::G;
  constexpr int NT = KGroup<KIND>::NT;
  static_assert(P1Layout<KIND>::END <= 2 * NT, "pass 1 fits two items per thread");
  constexpr int P2 = P2Layout<KIND>::END;
  static_assert(P2 <= 3 * NT, "pass 2 fits three items per thread");
  static_assert(G * NP <= NT, "pass 3 fits one point per thread");
  using Q = typename EvalPolicy<kind_of_kv(KIND), P>::type;
  constexpr bool kSort = sort_u<KIND>();
  constexpr int NU = Cache<KIND>::NU_TOTAL;
  const int ng = stage_regions<D, G, NT>(L, list, count, group, St);
  const int tid = threadIdx.x;
  const DevTables T = L.T;
  if (kSort && tid == 0) s_ucnt = 0;
  pass1<KIND, Q>(T, St, C, tid, ng);
  if constexpr (P1Layout<KIND>::END > NT) pass1<KIND, Q>(T, St, C, tid + NT, ng);
  __syncthreads();
  if constexpr (staged_p1<KIND>()) {
    static_assert(P1bLayout<KIND>::END <= 2 * NT, "pass 1b fits two items per thread");
    pass1b<KIND, Q>(T, St, C, tid, ng);
    if constexpr (P1bLayout<KIND>::END > NT) pass1b<KIND, Q>(T, St, C, tid + NT, ng);
    __syncthreads();
  }
  if constexpr (kSort) {
    constexpr int R = (P2 + NT - 1) / NT;
    uint16_t *ends = reinterpret_cast<uint16_t *>(s_f), *mid = ends + NU;
    sort_round<KIND, Q, 0, R>(T, St, C, tid, ng, &s_ucnt, s_unf, ends, mid);
    __syncthreads();
    const unsigned long long cw = s_ucnt;
    const uint32_t nb = (uint32_t)cw & 0x1fffffu, nbm = nb + ((uint32_t)(cw >> 21) & 0x1fffffu);
    const uint32_t nu = nbm + (uint32_t)(cw >> 42);
    // fixed rounds rather than a loop: in a loop the compiler keeps the
    // polynomial coefficients in registers across iterations and spills them
    constexpr int RU = (NU + NT - 1) / NT;
#pragma unroll
    for (int r = 0; r < RU; ++r) {
      const uint32_t j = tid + r * NT;
      if (j < nu) {
        const uint16_t item = j < nb ? ends[j] : j < nbm ? mid[j - nb] : ends[NU - 1 - (j - nbm)];
        u_eval_sorted<KIND, Q>(C, item, s_unf);
      }
    }
  } else {
    pass2<KIND, Q>(T, St, C, tid, ng);
    if constexpr (P2 > NT) pass2<KIND, Q>(T, St, C, tid + NT, ng);
    if constexpr (P2 > 2 * NT) pass2<KIND, Q>(T, St, C, tid + 2 * NT, ng);
  }
  __syncthreads();
  if (tid < ng * NP) {
    const int g = tid / NP, q = tid - g * NP;
    if (St.slot[g] != 0xffffffffu) {
      CachedSrc<KIND, Q> src(C, St.args[g], g, q);
      s_f[tid] = integrand_src<kind_of_kv(KIND), Q>(T, St.args[g], src);
    }
  }
  __syncthreads();
  reduce_regions<D, G, NP>(L, St, s_f, ng);
}

// At most 64 VGPRs (8 waves per SIMD): the FP64 5-D and 7-D kinds otherwise
// compile to 70-80 and run 6-7 waves per SIMD.  The few registers this
// spills cost less than the lost occupancy: NNMap 1h 4.12 -> 3.69 ms and
// 3h 4.26 -> 3.93 ms per launch on the 550-triplet workload, 2h unchanged.
template <int KIND, class P>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8))) void k_eval(EvalLaunch L) {
  // variables of their own, not one EvalLds: the compiler then knows them apart
  // (as one struct, 550 triplets took 262.8 ms rather than 261.6, the 2h kind most)
  using M = EvalLds<KIND>;
  __shared__ typename M::Stg St;
  __shared__ Cache<KIND> C;
  __shared__ double s_f[M::NF];
  __shared__ unsigned long long s_ucnt;
  __shared__ uint16_t s_unf[M::NUNF];
  const uint32_t group = block_group();
  if (group * KGroup<KIND>::G >= L.count) return;
  eval_block<KIND, P>(L, L.list, L.count, group, St, C, s_f, s_ucnt, s_unf);
}

// A whole round's evaluation in one launch, for small rounds (kSmallBlocks): the
// kinds run beside each other and fill the chip together instead of one after
// the other, each with its launch gap and its last wave of blocks, and the
// lists' lengths are read where the selection left them, so that the host can
// queue a round before it knows the last one's outcome.  Every kind in its
// 512-thread shape, which differs from the large rounds' only in speed.
template <int KIND>
struct SmallKv {
  static constexpr int kv = make_kv(KIND, kind_dim(KIND) == 6 ? 3 : 1);
  static_assert(KGroup<kv>::NT == kSmallThreads, "one block size for all kinds");
};
template <int KIND>
__device__ __forceinline__ void eval_small(const EvalSmallLaunch &L, uint32_t group,
                                           unsigned char *lds) {
  constexpr int kv = SmallKv<KIND>::kv;
  const uint32_t count = L.row ? L.row[KIND] : L.count[KIND];
  if (group * KGroup<kv>::G >= count) return;
  EvalLds<kv> &M = *reinterpret_cast<EvalLds<kv> *>(lds);
  eval_block<kv, P64>(L.E, L.lists[KIND], count, group, M.St, M.C, M.f, M.ucnt, M.unf);
  if (L.clock && threadIdx.x == 0)
    atomicMax(reinterpret_cast<unsigned long long *>(L.clock) + kRowKindEnd + KIND,
              (unsigned long long)wall_clock64());
}
__global__ __launch_bounds__(kSmallThreads) __attribute__((amdgpu_waves_per_eu(8))) void
k_eval_small(EvalSmallLaunch L) {
  constexpr size_t a = sizeof(EvalLds<SmallKv<kNN1>::kv>), b = sizeof(EvalLds<SmallKv<kNN2>::kv>),
                   c = sizeof(EvalLds<SmallKv<kNN3>::kv>), d = sizeof(EvalLds<SmallKv<kNM1>::kv>),
                   e = sizeof(EvalLds<SmallKv<kNM2>::kv>), f = sizeof(EvalLds<SmallKv<kNM3>::kv>);
  constexpr size_t ab = a > b ? a : b, cd = c > d ? c : d, ef = e > f ? e : f,
                   abcd = ab > cd ? ab : cd;
  __shared__ __align__(16) unsigned char lds[abcd > ef ? abcd : ef];
  const uint32_t bl = blockIdx.x;
  if (L.clock && bl == 0 && threadIdx.x == 0) L.clock[kRowStart] = (uint64_t)wall_clock64();
  if (bl < L.end[kNN1]) eval_small<kNN1>(L, bl, lds);
  else if (bl < L.end[kNN2]) eval_small<kNN2>(L, bl - L.end[kNN1], lds);
  else if (bl < L.end[kNN3]) eval_small<kNN3>(L, bl - L.end[kNN2], lds);
  else if (bl < L.end[kNM1]) eval_small<kNM1>(L, bl - L.end[kNN3], lds);
  else if (bl < L.end[kNM2]) eval_small<kNM2>(L, bl - L.end[kNM1], lds);
  else eval_small<kNM3>(L, bl - L.end[kNM2], lds);
}
uint32_t small_group(int kind) {
  const int d = kind_dim(kind);
  return d == 5 ? KGroup<SmallKv<kNN1>::kv>::G
                : d == 6 ? KGroup<SmallKv<kNN2>::kv>::G : KGroup<SmallKv<kNN3>::kv>::G;
}
hipError_t launch_eval_small(const EvalSmallLaunch &L, hipStream_t s) {
  const uint32_t blocks = L.end[kNumKinds - 1];
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_eval_small, dim3(blocks), dim3(kSmallThreads), 0, s, L);
  return hipGetLastError();
}

// ----------------------------------------------------------------- roots
__device__ __forceinline__ double box_volume(int D, const double *h) {
  double v = 1;
  for (int i = 0; i < D; ++i) v *= 2 * h[i];
  return v;
}

__global__ void k_roots(RootsLaunch L) {
  uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= L.njobs) return;
  JobDesc d = L.jobs[j];
  const double *lo = L.boxes + (size_t)j * 2 * kMaxDim;
  const double *hi = lo + kMaxDim;
  const uint64_t S = L.stride;
  double h[kMaxDim];
  for (int i = 0; i < d.dim; ++i) {
    double c = 0.5 * (lo[i] + hi[i]);
    h[i] = 0.5 * (hi[i] - lo[i]);
    L.geo[(kFieldC + i) * S + d.base] = c;
    L.geo[(kFieldH + i) * S + d.base] = h[i];
  }
  L.geo[kFieldVol * S + d.base] = box_volume(d.dim, h);
  L.split[d.base] = 0;
  JobState st;
  st.neval = (uint64_t)d.pts;
  st.n = 1;
  st.flags = 0;
  st.rounds = 0;
  st.pad = 0;
  st.val = 0;
  st.err = 0;
  L.state[j] = st;
  uint32_t at = atomicAdd(&L.counters[d.kind], 1u);
  L.lists[d.kind][at] = EvalItem{d.base, j};
}

__global__ void k_admit(AdmitLaunch L) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= L.n) return;
  const uint32_t j = L.ids[t];
  const JobDesc d = L.desc[t];
  L.jobs[j] = d;
  L.args_table[j] = L.args[t];
  const double *lo = L.boxes + (size_t)t * 2 * kMaxDim;
  const double *hi = lo + kMaxDim;
  const uint64_t S = L.stride;
  double h[kMaxDim];
  for (int i = 0; i < d.dim; ++i) {
    double c = 0.5 * (lo[i] + hi[i]);
    h[i] = 0.5 * (hi[i] - lo[i]);
    L.geo[(kFieldC + i) * S + d.base] = c;
    L.geo[(kFieldH + i) * S + d.base] = h[i];
  }
  L.geo[kFieldVol * S + d.base] = box_volume(d.dim, h);
  L.split[d.base] = 0;
  JobState st;
  st.neval = (uint64_t)d.pts;
  st.n = 1;
  st.flags = 0;
  st.rounds = 0;
  st.pad = 0;
  st.val = 0;
  st.err = 0;
  L.state[j] = st;
  uint32_t at = atomicAdd(&L.counters[d.kind], 1u);
  L.lists[d.kind][at] = EvalItem{d.base, j};
}

__global__ void k_gather(GatherLaunch L) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < L.n) L.out[t] = L.state[L.ids[t]];
}

// The index argument of the mass coordinates' centre (DevTables::xc_ix) to out.
__global__ void k_mass_centre(DevTables T, double *out) {
  double m, L;
  *out = mass_chain(T, T.xc(), m, L);
}
hipError_t launch_mass_centre(const DevTables &T, double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_mass_centre, dim3(1), dim3(1), 0, s, T, out);
  return hipGetLastError();
}

__global__ void k_zero(uint32_t *p, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ---------------------------------------------------------------- select
// One block per integral: totals, stop tests, the Gladwell batch and its cuts.
// It is bound by latency -- passes over the integral's errors in memory, with
// few bytes each -- so the passes are few (totals; a histogram; the keys near
// the batch's boundary; the cuts) and wide: 1024 threads per integral up to
// kSelectWideJobs integrals, 256 beyond.  Up to 256 regions one wave does it
// all, from registers and without a barrier.  An earlier form with 256 threads
// and eight radix levels, each a pass over the errors, took 2.47 ms for a run
// of 9 integrals and 6.9 ms for 1650 (now 1.11 and 5.2).
//
// Both thread counts and the one-wave form add in the same order and select by
// the same rule: an integral's result does not depend on which of them runs.

// The totals' order: 256 partial sums over i = t, t + 256, ..., then pairwise
// (t, t + 128), (t, t + 64), ..., (0, 1); value compensated, error plain.
constexpr int kPartial = 256;

template <int NT>
struct SelectLds {
  JobState st;
  double vs[kPartial], vc[kPartial], es[kPartial];
  uint64_t kmax[NT / 64];
  uint32_t bad;
  // histogram of the keys' distance below the largest, eight bins per octave
  unsigned long long sum[256];
  uint32_t cnt[256];
  uint64_t lo, width;            // the bin that holds the boundary
  uint32_t m, above;
  unsigned long long rest;
  // candidates: keys of that bin
  uint64_t key[1024];
  uint32_t nkey;
  double bs[NT / 64], bc[NT / 64];
  uint32_t wcnt[NT / 64], wtie[NT / 64];
  SearchLds search;
  Boundary B;
  double V, E;
  uint64_t maxkey;
  int found, stop;
  uint32_t listbase;
  uint32_t sel[4 * NT];          // slots cut in one chunk, ascending
};

// Ends a job's selection: state to memory, the job to the done list.
__device__ __forceinline__ void select_finish(const SelectLaunch &L, uint32_t J, const JobState &st) {
  L.state[J] = st;
  if (L.done) L.done[atomicAdd(&L.counters[kNumKinds + 1], 1u)] = J;
}

// Stop tests in the order of src/hcubature.cpp:938-939 on totals (V, E).
__device__ __forceinline__ bool select_stops(const JobDesc &d, double V, double E, bool nonfinite,
                                             JobState &st) {
  st.val = V;
  st.err = E;
  if (nonfinite) st.flags |= kJobNonfinite;
  if (d.maxeval != 0 && st.neval >= d.maxeval) {
    st.flags |= kJobDone | kJobCapped;
    return true;
  }
  if (!(E > 0 && E > fabs(V) * d.reltol)) {
    st.flags |= kJobDone | kJobConverged;
    return true;
  }
  return false;
}

// The most regions the evaluation budget lets a batch pop.
__device__ __forceinline__ uint64_t select_kcap(const JobDesc &d, const JobState &st) {
  if (d.maxeval == 0) return st.n;
  const uint64_t twoP = 2ull * (uint64_t)d.pts, room = d.maxeval - st.neval;
  const uint64_t kc = (room + twoP - 1) / twoP;
  return kc < st.n ? kc : st.n;
}

// Room for a batch of K regions: its place in the kind's list, or false when
// the integral's slots or the list are full.  One thread calls it.
__device__ __forceinline__ bool select_room(const SelectLaunch &L, const JobDesc &d, uint32_t K,
                                            JobState &st, uint32_t &listbase) {
  if (st.n + K > d.cap) {
    st.flags |= kJobDone | kJobPoolFull;
    return false;
  }
  listbase = atomicAdd(&L.counters[d.kind], 2u * K);
  if (listbase + 2u * K > L.list_cap[d.kind]) {
    st.flags |= kJobDone | kJobPoolFull;
    return false;
  }
  atomicAdd(&L.counters[kNumKinds], 1u);
  return true;
}

// Cuts the region in slot p along its split dimension, the a-th region of a
// batch of K: the lower half keeps the slot, the upper one goes to slot q.  The
// list holds the K kept slots first and the K new ones after them, both in
// slot order, so that the regions an evaluation block stages sit in
// neighbouring slots of each field.
__device__ __forceinline__ void select_cut(const SelectLaunch &L, EvalItem *list, uint32_t J, int D,
                                           uint32_t p, uint32_t q, uint32_t a, uint32_t K) {
  const uint64_t S = L.stride;
  const int sd = L.split[p];
  double c[kMaxDim], h[kMaxDim], hd = 0;
#pragma unroll
  for (int e = 0; e < kMaxDim; ++e) {
    if (e < D) {
      c[e] = L.geo[(kFieldC + e) * S + p];
      h[e] = L.geo[(kFieldH + e) * S + p];
    }
  }
#pragma unroll
  for (int e = 0; e < kMaxDim; ++e)
    if (e < D && e == sd) hd = h[e] * 0.5;
  const double vol = L.geo[kFieldVol * S + p];
  double vq = 1;  // box_volume of the new half, the same products in order
#pragma unroll
  for (int e = 0; e < kMaxDim; ++e) {
    if (e >= D) continue;
    const double he = (e == sd) ? hd : h[e];
    vq *= 2 * he;
    L.geo[(kFieldC + e) * S + q] = (e == sd) ? c[e] + hd : c[e];
    L.geo[(kFieldH + e) * S + q] = he;
    if (e == sd) {
      L.geo[(kFieldC + e) * S + p] = c[e] - hd;
      L.geo[(kFieldH + e) * S + p] = hd;
    }
  }
  L.geo[kFieldVol * S + p] = vol * 0.5;
  L.geo[kFieldVol * S + q] = vq;
  list[a] = EvalItem{p, J};
  list[K + a] = EvalItem{q, J};
}

// The job's state after a batch of K regions.  One thread calls it.
__device__ __forceinline__ void select_commit(const SelectLaunch &L, const JobDesc &d, uint32_t J,
                                              uint32_t K, JobState st) {
  if (L.trace && st.rounds < L.trace_cap) L.trace[(size_t)J * L.trace_cap + st.rounds] = 2u * K;
  st.n += K;
  st.neval += 2ull * (uint64_t)d.pts * K;
  st.rounds += 1;
  L.state[J] = st;
}

// n <= 64 R regions by one wave.
template <int R>
__device__ __forceinline__ void select_wave(const SelectLaunch &L, uint32_t J, const JobDesc &d,
                                            JobState st, SearchLds &W, uint32_t *list_p) {
  const int lane = threadIdx.x & 63;
  const uint32_t n = st.n;
  const uint64_t S = L.stride;
  const double *val = L.geo + kFieldVal * S + d.base, *err = L.geo + kFieldErr * S + d.base;
  uint64_t k[R];
  double v[R], e[R], c[R], check = 0;
  uint64_t maxkey = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t i = 64 * r + lane;
    v[r] = i < n ? val[i] : 0.0;
    e[r] = i < n ? err[i] : 0.0;
    c[r] = 0;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    check = fma(0.0, v[r], fma(0.0, e[r], check));
    const uint64_t ke = err_key(e[r]);
    k[r] = 64u * r + lane < n ? ke : ~0ull;
    maxkey = ke > maxkey ? ke : maxkey;
  }
#pragma unroll
  for (int w = R / 2; w > 0; w >>= 1) {
#pragma unroll
    for (int q = 0; q < w; ++q) {
      const double t = v[q] + v[q + w];
      c[q] += c[q + w] + sum_error(v[q], v[q + w], t);
      v[q] = t;
      e[q] += e[q + w];
    }
  }
  const double V = comp_total(v[0], c[0]);
  double E = e[0];
  tree([&](auto w) { E += from_above<decltype(w)::value>(E); });
  E = readlane64(E, 0);
  if (select_stops(d, V, E, __ballot(check != check) != 0, st)) {
    if (lane == 0) select_finish(L, J, st);
    return;
  }
  // every key is among these, so the boundary is
  Boundary B{};
  (void)find_boundary<R>(k, n, wave_max(maxkey), Goal{fabs(V) * d.reltol, select_kcap(d, st), 0, 0.0},
                         W, B);
  const uint32_t K = B.gt + B.take;
  uint32_t listbase = 0, ok = 0;
  if (lane == 0) ok = select_room(L, d, K, st, listbase) ? 1u : 0u;
  listbase = __builtin_amdgcn_readfirstlane(listbase);
  if (!__builtin_amdgcn_readfirstlane(ok)) {
    if (lane == 0) select_finish(L, J, st);
    return;
  }
  uint32_t at = 0, ties = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const bool in = k[r] != ~0ull, tie = in && k[r] == B.T;
    const uint64_t tm = __ballot(tie);
    const bool s = in && (k[r] > B.T || (tie && ties + lanes_below(tm) < B.take));
    ties += (uint32_t)__popcll(tm);
    const uint64_t sm = __ballot(s);
    if (s) list_p[at + lanes_below(sm)] = 64 * r + lane;
    at += (uint32_t)__popcll(sm);
  }
  wave_sync();
  EvalItem *list = L.lists[d.kind] + listbase;
  for (uint32_t a = lane; a < K; a += 64)
    select_cut(L, list, J, d.dim, d.base + list_p[a], d.base + n + a, a, K);
  if (lane == 0) select_commit(L, d, J, K, st);
}

// Whether popping every key >= T of the integral is enough, over the whole
// block (the bisection's test).
template <int NT>
__device__ bool block_enough(const double *err, uint32_t n, uint64_t T, const Goal &g,
                             SelectLds<NT> &S, uint32_t &ge) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double s = 0, c = 0;
  uint32_t cnt = 0;
  for (uint32_t i = tid; i < n; i += NT) {
    const uint64_t k = err_key(err[i]);
    comp_add(s, c, k < T ? __builtin_bit_cast(double, k) : 0.0);
    cnt += k >= T;
  }
  comp_tree(s, c);
  tree([&](auto w) { cnt += from_above32<decltype(w)::value>(cnt); });
  __syncthreads();
  if (lane == 0) {
    S.bs[wave] = s;
    S.bc[wave] = c;
    S.wcnt[wave] = cnt;
  }
  __syncthreads();
  double ts = 0, tc = 0;
  ge = 0;
  for (int w = 0; w < NT / 64; ++w) {
    comp_add(ts, tc, S.bs[w]);
    tc += S.bc[w];
    ge += S.wcnt[w];
  }
  return ge >= g.kcap || meets(ts + tc, g.thr);
}

template <int NT>
__device__ __forceinline__ void select_block(const SelectLaunch &L, uint32_t J, const JobDesc &d,
                                             SelectLds<NT> &S) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint64_t St = L.stride;
  const uint32_t n = S.st.n;
  const double *val = L.geo + kFieldVal * St + d.base, *err = L.geo + kFieldErr * St + d.base;
  constexpr int U = 8;   // loads in flight per thread

  // 1. totals.  With 1024 threads the first four waves take the values and the
  //    next four the errors.
  const bool tv = tid < kPartial, te = NT == kPartial ? true : (tid >= kPartial && tid < 2 * kPartial);
  double check = 0;
  uint64_t kmax = 0;
  if (tv) {
    double s = 0, c = 0;
    for (uint32_t i0 = tid; i0 < n; i0 += U * kPartial) {
      double v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = i0 + u * kPartial < n ? val[i0 + u * kPartial] : 0.0;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        check = fma(0.0, v[u], check);
        comp_add(s, c, v[u]);
      }
    }
    S.vs[tid] = s;
    S.vc[tid] = c;
  }
  if (te) {
    const int t = tid & (kPartial - 1);
    double s = 0;
    for (uint32_t i0 = t; i0 < n; i0 += U * kPartial) {
      double e[U];
#pragma unroll
      for (int u = 0; u < U; ++u) e[u] = i0 + u * kPartial < n ? err[i0 + u * kPartial] : 0.0;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        check = fma(0.0, e[u], check);
        s += e[u];
        const uint64_t k = err_key(e[u]);
        kmax = k > kmax ? k : kmax;
      }
    }
    S.es[t] = s;
    kmax = wave_max(kmax);
    if (lane == 0) S.kmax[(tid & (kPartial - 1)) >> 6] = kmax;
  }
  if (__ballot(check != check) != 0 && lane == 0) atomicOr(&S.bad, 1u);
  if (tid < 256) {
    S.sum[tid] = 0;
    S.cnt[tid] = 0;
  }
  __syncthreads();
  if (wave == 0) {
    double s[4], c[4], e[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      s[q] = S.vs[64 * q + lane];
      c[q] = S.vc[64 * q + lane];
      e[q] = S.es[64 * q + lane];
    }
#pragma unroll
    for (int w = 2; w > 0; w >>= 1) {
#pragma unroll
      for (int q = 0; q < w; ++q) {
        const double t = s[q] + s[q + w];
        c[q] += c[q + w] + sum_error(s[q], s[q + w], t);
        s[q] = t;
        e[q] += e[q + w];
      }
    }
    const double V = comp_total(s[0], c[0]);
    double E = e[0];
    tree([&](auto w) { E += from_above<decltype(w)::value>(E); });
    E = readlane64(E, 0);
    if (lane == 0) {
      uint64_t k = S.kmax[0];
      for (int w = 1; w < kPartial / 64; ++w) k = S.kmax[w] > k ? S.kmax[w] : k;
      S.maxkey = k;
      S.V = V;
      S.E = E;
      // 2. stop tests
      JobState st = S.st;
      S.stop = select_stops(d, V, E, S.bad != 0, st) ? 1 : 0;
      S.st = st;
      if (S.stop) select_finish(L, J, st);
      S.lo = 0;
      S.width = 1ull << 63;
      S.above = 0;
      S.rest = 0;
      S.nkey = 0;
      S.found = 0;
    }
  }
  __syncthreads();
  if (S.stop) return;

  // 3. the batch's boundary.  A histogram pass names the bin that holds it
  //    (narrowed while the bin has more keys than fit LDS), a second pass
  //    collects that bin's keys and sums the smaller ones exactly, and the
  //    first wave finds the boundary among them.
  const uint64_t maxkey = S.maxkey;
  const Goal goal{fabs(S.V) * d.reltol, select_kcap(d, S.st), 0, 0.0};
  const int shift = sel_shift(maxkey, n);
  const double thr_fx = ldexp(goal.thr, shift);
  int s = 49;
  for (;;) {
    const uint64_t lo = S.lo, width = S.width;
    for (uint32_t i0 = tid; i0 < n; i0 += 4 * NT) {
      double e[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) e[u] = i0 + u * NT < n ? err[i0 + u * NT] : 0.0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint64_t k = err_key(e[u]), dd = maxkey - k - lo;
        if (i0 + u * NT < n && k <= maxkey - lo && dd < width) {
          const uint64_t q = dd >> s;
          const int b = q < 255 ? (int)q : 255;
          atomicAdd(&S.cnt[b], 1u);
          atomicAdd(&S.sum[b], fixed_err(k, shift));
        }
      }
    }
    __syncthreads();
    if (wave == 0) {
      // lane l takes bins 4 l .. 4 l + 3
      unsigned long long bsum[4], own = 0;
      uint32_t bcnt[4], cown = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        bsum[q] = S.sum[4 * lane + q];
        bcnt[q] = S.cnt[4 * lane + q];
        own += bsum[q];
        cown += bcnt[q];
      }
      unsigned long long suf = own;
      uint32_t pre = cown;
#pragma unroll
      for (int w = 1; w < 64; w <<= 1) {
        const uint32_t l2 = __shfl_down((uint32_t)suf, w), h2 = __shfl_down((uint32_t)(suf >> 32), w);
        const uint32_t p2 = __shfl_up(pre, w);
        if (lane + w < 64) suf += ((unsigned long long)h2 << 32) | l2;
        if (lane >= w) pre += p2;
      }
      // the first non-empty bin after which enough is popped, else the last one
      unsigned long long rest = suf + S.rest;     // remaining before this lane's bins
      uint32_t cum = S.above + pre - cown;        // popped before them
      int first = -1, last = -1;
      uint32_t cfirst = 0, clast = 0;
      unsigned long long rfirst = 0, rlast = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        rest -= bsum[q];
        if (bcnt[q]) {
          if (first < 0 && ((double)rest <= thr_fx || (uint64_t)cum + bcnt[q] >= goal.kcap)) {
            first = q;
            cfirst = cum;
            rfirst = rest;
          }
          last = q;
          clast = cum;
          rlast = rest;
        }
        cum += bcnt[q];
      }
      const uint64_t hit = __ballot(first >= 0), some = __ballot(last >= 0);
      const int who = hit ? __ffsll((unsigned long long)hit) - 1 : 63 - __clzll((long long)some);
      if (lane == who) {
        const int q = hit ? first : last;
        const int b = 4 * lane + q;
        S.above = hit ? cfirst : clast;
        S.rest = hit ? rfirst : rlast;
        uint32_t mq = 0;
#pragma unroll
        for (int x = 0; x < 4; ++x) mq = x == q ? bcnt[x] : mq;
        S.m = mq;
        S.lo = lo + ((uint64_t)b << s);
        S.width = b == 255 ? width - ((uint64_t)255 << s) : 1ull << s;
      }
    }
    __syncthreads();
    if (S.m <= 1024 || S.width <= 1) break;
    s = 56 - __clzll((long long)(S.width - 1));   // ceil(log2 width) - 8
    s = s < 0 ? 0 : s;
    if (tid < 256) {
      S.sum[tid] = 0;
      S.cnt[tid] = 0;
    }
    __syncthreads();
  }
  {
    const uint64_t khi = maxkey - S.lo, w1 = S.width - 1, klo = khi >= w1 ? khi - w1 : 0;
    const bool few = S.m <= 1024;
    double bs = 0, bc = 0;
    for (uint32_t i0 = tid; i0 < n; i0 += 4 * NT) {
      double e[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) e[u] = i0 + u * NT < n ? err[i0 + u * NT] : 0.0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint64_t k = err_key(e[u]);
        comp_add(bs, bc, k < klo ? __builtin_bit_cast(double, k) : 0.0);
        if (few && i0 + u * NT < n && k >= klo && k <= khi) S.key[atomicAdd(&S.nkey, 1u)] = k;
      }
    }
    comp_tree(bs, bc);
    if (lane == 0) {
      S.bs[wave] = bs;
      S.bc[wave] = bc;
    }
    __syncthreads();
    if (wave == 0) {
      double ts = 0, tc = 0;
      for (int w = 0; w < NT / 64; ++w) {
        comp_add(ts, tc, S.bs[w]);
        tc += S.bc[w];
      }
      Goal g = goal;
      g.above = S.above;
      g.below = ts + tc;
      const uint32_t m = S.m;
      Boundary B{};
      bool ok;
      auto search = [&](auto tag) {
        constexpr int R = decltype(tag)::value;
        uint64_t k[R], km = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const uint32_t i = 64 * r + lane;
          k[r] = i < m ? S.key[i] : ~0ull;
          km = i < m && k[r] > km ? k[r] : km;
        }
        return find_boundary<R>(k, m, wave_max(km), g, S.search, B);
      };
      if (!few) {   // one key, many regions
        const double all = g.below + (double)m * __builtin_bit_cast(double, khi);
        ok = (meets(g.below, g.thr) || (uint64_t)g.above + m >= g.kcap) &&
             (g.above == 0 || !(meets(all, g.thr) || g.above >= g.kcap));
        B = Boundary{khi, m, fewest(g, khi, m, g.above, g.below), g.above};
      } else if (m <= 64) {
        ok = search(Int<1>{});
      } else if (m <= 256) {
        ok = search(Int<4>{});
      } else {
        ok = search(Int<16>{});
      }
      if (lane == 0) {
        S.found = ok ? 1 : 0;
        S.B = B;
      }
    }
    __syncthreads();
  }
  if (!S.found) {
    // the truncated sums named the wrong bin: bisection over the key's bits
    uint64_t t = 0;
    uint32_t ge = 0;
    for (int bit = 62; bit >= 0; --bit) {
      const uint64_t u = t | (1ull << bit);
      if (u <= maxkey && block_enough<NT>(err, n, u, goal, S, ge)) t = u;
    }
    (void)block_enough<NT>(err, n, t, goal, S, ge);
    uint32_t more = 0;
    (void)block_enough<NT>(err, n, t + 1, goal, S, more);
    // the sum below t once more, for the multiplicity's share
    double ts = 0, tc = 0;
    for (uint32_t i = tid; i < n; i += NT) {
      const uint64_t k = err_key(err[i]);
      comp_add(ts, tc, k < t ? __builtin_bit_cast(double, k) : 0.0);
    }
    comp_tree(ts, tc);
    __syncthreads();
    if (lane == 0) {
      S.bs[wave] = ts;
      S.bc[wave] = tc;
    }
    __syncthreads();
    if (tid == 0) {
      double a = 0, b = 0;
      for (int w = 0; w < NT / 64; ++w) {
        comp_add(a, b, S.bs[w]);
        b += S.bc[w];
      }
      S.B = Boundary{t, ge - more, fewest(goal, t, ge - more, more, a + b), more};
    }
    __syncthreads();
  }
  const Boundary B = S.B;
  const uint32_t K = B.gt + B.take;
  if (tid == 0) {
    JobState st = S.st;
    S.stop = select_room(L, d, K, st, S.listbase) ? 0 : 1;
    if (S.stop) select_finish(L, J, st);
  }
  __syncthreads();
  if (S.stop) return;

  // 4. the cuts, in slot order: each thread looks at four consecutive slots of
  //    a chunk; ranks among the batch (and, where only part of the regions at
  //    T go, among those) come from wave scans and the waves' totals, and the
  //    chunk's slots are listed in LDS in rank order, so that consecutive
  //    lanes cut consecutive regions.
  EvalItem *list = L.lists[d.kind] + S.listbase;
  const bool some_ties = B.take != B.eq;
  uint32_t done = 0, ties = 0;
  for (uint32_t chunk = 0; chunk < n; chunk += 4 * NT) {
    const uint32_t i0 = chunk + 4 * tid;
    uint64_t k[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) k[u] = i0 + u < n ? err_key(err[i0 + u]) : 0;
    uint32_t selm = 0, tiem = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool in = i0 + u < n;
      selm |= in && (some_ties ? k[u] > B.T : k[u] >= B.T) ? 1u << u : 0u;
      tiem |= in && k[u] == B.T ? 1u << u : 0u;
    }
    auto scan = [&](uint32_t own, uint32_t *w_tot, uint32_t &total) {
      uint32_t inc = own;
#pragma unroll
      for (int w = 1; w < 64; w <<= 1) {
        const uint32_t x = __shfl_up(inc, w);
        if (lane >= w) inc += x;
      }
      if (lane == 63) w_tot[wave] = inc;
      __syncthreads();
      uint32_t before = 0;
      total = 0;
#pragma unroll
      for (int w = 0; w < NT / 64; ++w) {
        const uint32_t x = w_tot[w];
        before += w < wave ? x : 0u;
        total += x;
      }
      return before + inc - own;
    };
    if (some_ties) {
      uint32_t tot, rank = ties + scan((uint32_t)__popc(tiem), S.wtie, tot);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (tiem >> u & 1u) {
          selm |= rank < B.take ? 1u << u : 0u;
          ++rank;
        }
      ties += tot;
    }
    uint32_t tot, at = scan((uint32_t)__popc(selm), S.wcnt, tot);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (selm >> u & 1u) S.sel[at++] = i0 + u;
    __syncthreads();
    for (uint32_t j = tid; j < tot; j += NT)
      select_cut(L, list, J, d.dim, d.base + S.sel[j], d.base + n + done + j, done + j, K);
    done += tot;
    __syncthreads();
  }
  if (tid == 0) select_commit(L, d, J, K, S.st);
}

template <int NT>
__global__ __launch_bounds__(NT) void k_select(SelectLaunch L) {
  __shared__ SelectLds<NT> S;
  const uint32_t J = L.active ? L.active[blockIdx.x] : blockIdx.x;
  // through LDS: the last act of the block's first thread is a new state
  if (threadIdx.x == 0) {
    S.st = L.state[J];
    S.bad = 0;
  }
  __syncthreads();
  if (L.clock && blockIdx.x == 0 && threadIdx.x == 0) L.clock[kRowSelect] = (uint64_t)wall_clock64();
  if (S.st.flags & kJobDone) return;
  const JobDesc d = L.jobs[J];
  if (S.st.n <= 256) {
    if (threadIdx.x >= 64) return;
    if (S.st.n <= 64) select_wave<1>(L, J, d, S.st, S.search, S.sel);
    else select_wave<4>(L, J, d, S.st, S.search, S.sel);
  } else {
    select_block<NT>(L, J, d, S);
  }
  if (L.clock && threadIdx.x == 0)
    atomicMax(reinterpret_cast<unsigned long long *>(L.clock) + kRowSelectEnd,
              (unsigned long long)wall_clock64());
}


// ---------------------------------------------------------- point values
// The integrand at caller-given points x[npts][dim] (one thread per point),
// the device counterpart of the reference's integrand callbacks.
template <int KIND, class P>
__global__ void k_points(DevTables T, const TermArgs *args, const double *x, uint32_t npts,
                         double *f) {
  constexpr int D = kind_dim(kind_of_kv(KIND));
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npts) return;
  double p[D];
#pragma unroll
  for (int d = 0; d < D; ++d) p[d] = x[(size_t)i * D + d];
  f[i] = integrand<KIND, P>(T, *args, p);
}

template <class P>
static void points_kind(int kind, dim3 g, dim3 b, hipStream_t s, const DevTables &T,
                        const TermArgs *args, const double *x, uint32_t npts, double *f) {
  switch (kind) {
    case kNbar: hipLaunchKernelGGL((k_points<kNbar, P>), g, b, 0, s, T, args, x, npts, f); break;
    case kNN1: hipLaunchKernelGGL((k_points<kNN1, P>), g, b, 0, s, T, args, x, npts, f); break;
    case kNN2: hipLaunchKernelGGL((k_points<kNN2, P>), g, b, 0, s, T, args, x, npts, f); break;
    case kNN3: hipLaunchKernelGGL((k_points<kNN3, P>), g, b, 0, s, T, args, x, npts, f); break;
    case kNM1: hipLaunchKernelGGL((k_points<kNM1, P>), g, b, 0, s, T, args, x, npts, f); break;
    case kNM2: hipLaunchKernelGGL((k_points<kNM2, P>), g, b, 0, s, T, args, x, npts, f); break;
    default: hipLaunchKernelGGL((k_points<kNM3, P>), g, b, 0, s, T, args, x, npts, f); break;
  }
}

hipError_t launch_points(int kind, int prec, const DevTables &T, const TermArgs *args,
                         const double *x, uint32_t npts, double *f, hipStream_t s) {
  if (npts == 0) return hipSuccess;
  if (kind < 0 || kind >= kNumKinds) return hipErrorInvalidValue;
  dim3 g((npts + 255) / 256), b(256);
  if (prec == 0 || kind == kNbar) points_kind<P64>(kind, g, b, s, T, args, x, npts, f);
  else points_kind<PMix>(kind, g, b, s, T, args, x, npts, f);
  return hipGetLastError();
}

// ------------------------------------------------- precomputation tables
// The closed-form 2-D tables of the precomputation from its integrals, one
// thread per (z, m or k) entry: linear P(k, z) (src/Powerspectrum.cpp:200-207),
// c(m, z) = 9/(1+z) (m/m*)^-0.13 (:128-135), the Sheth-Tormen mass function
// and bias (src/HMF.cpp:7-49, with pi = 3.14159 of src/constants.h:15).
__global__ void k_precomp_tables(PrecompTablesLaunch L) {
  const int n = L.nb * L.nb;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int iz = i / L.nb, j = i - iz * L.nb;
  const PrecompParams &p = *reinterpret_cast<const PrecompParams *>(L.aux);
  const double z = L.zs[iz], m = L.ms[j];
  L.plin[i] = eh_spectrum(p, L.ks[j], L.growth[iz]);
  const double c0 = 9, alpha = 0.13;
  L.conc[i] = c0 / (1. + z) * pow(m / L.mstar[iz], -alpha);
  const double A = 0.322, q = 0.707, pp = 0.3, pi = 3.14159;
  const double sigma2 = L.sigma2[i], dsigma2 = L.dsigma2[i], delta_c = L.delta_c[iz];
  const double rho_mean = L.rho_mean[iz];
  const double nuSq = delta_c * delta_c / sigma2;
  L.hmf[i] = -rho_mean / m / sigma2 * dsigma2 * A * (1 + pow(q * nuSq, -pp)) *
             sqrt(q * nuSq / 2 / pi) * exp(-0.5 * q * nuSq);
  L.bh[i] = 1 + 1. / delta_c *
                    (q * delta_c * delta_c / sigma2 - 1 +
                     2 * pp / (1 + pow(q * delta_c * delta_c / sigma2, pp)));
}

hipError_t launch_precomp_tables(const PrecompTablesLaunch &L, hipStream_t s) {
  const int n = L.nb * L.nb;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_precomp_tables, dim3((n + 255) / 256), dim3(256), 0, s, L);
  return hipGetLastError();
}

// ----------------------------------------------------------------- launch
template <int KV, class P>
static hipError_t launch_eval_kind(const EvalLaunch &L, hipStream_t s) {
  using Gr = KGroup<KV>;
  uint32_t blocks = (L.count + Gr::G - 1) / Gr::G;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL((k_eval<KV, P>), dim3(blocks), dim3(Gr::NT), 0, s, L);
  return hipGetLastError();
}

template <int V, class P>
static hipError_t launch_eval_variant(int kind, const EvalLaunch &L, hipStream_t s) {
  switch (kind) {
    case kNN1: return launch_eval_kind<make_kv(kNN1, V), P>(L, s);
    case kNN2: return launch_eval_kind<make_kv(kNN2, V), P>(L, s);
    case kNN3: return launch_eval_kind<make_kv(kNN3, V), P>(L, s);
    case kNM1: return launch_eval_kind<make_kv(kNM1, V), P>(L, s);
    case kNM2: return launch_eval_kind<make_kv(kNM2, V), P>(L, s);
    case kNM3: return launch_eval_kind<make_kv(kNM3, V), P>(L, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_eval(int kind, int prec, int variant, const EvalLaunch &L, hipStream_t s) {
  if (variant < 0 || variant >= kNumVariants) return hipErrorInvalidValue;
  if (prec == 0) {
    if (variant == 3) return launch_eval_variant<3, P64>(kind, L, s);
    if (variant == 2) return launch_eval_variant<2, P64>(kind, L, s);
    return variant ? launch_eval_variant<1, P64>(kind, L, s) : launch_eval_variant<0, P64>(kind, L, s);
  }
  if (variant == 3) return launch_eval_variant<3, PMix>(kind, L, s);
  if (variant == 2) return launch_eval_variant<2, PMix>(kind, L, s);
  return variant ? launch_eval_variant<1, PMix>(kind, L, s) : launch_eval_variant<0, PMix>(kind, L, s);
}

int eval_num_variants() { return kNumVariants; }

// Kernel symbols and block shapes, for launches recorded in a graph.
template <int KV, class P>
static KernelRef eval_ref_kind() {
  using Gr = KGroup<KV>;
  KernelRef r;
  r.fn = reinterpret_cast<const void *>(&k_eval<KV, P>);
  r.threads = (unsigned)Gr::NT;
  r.group = (unsigned)Gr::G;
  return r;
}

template <int V, class P>
static int eval_ref_variant(int kind, KernelRef *out) {
  switch (kind) {
    case kNN1: *out = eval_ref_kind<make_kv(kNN1, V), P>(); return 0;
    case kNN2: *out = eval_ref_kind<make_kv(kNN2, V), P>(); return 0;
    case kNN3: *out = eval_ref_kind<make_kv(kNN3, V), P>(); return 0;
    case kNM1: *out = eval_ref_kind<make_kv(kNM1, V), P>(); return 0;
    case kNM2: *out = eval_ref_kind<make_kv(kNM2, V), P>(); return 0;
    case kNM3: *out = eval_ref_kind<make_kv(kNM3, V), P>(); return 0;
    default: return -1;
  }
}

int eval_kernel_ref(int kind, int prec, int variant, KernelRef *out) {
  if (variant < 0 || variant >= kNumVariants) return -1;
  if (prec == 0) {
    if (variant == 3) return eval_ref_variant<3, P64>(kind, out);
    if (variant == 2) return eval_ref_variant<2, P64>(kind, out);
    return variant ? eval_ref_variant<1, P64>(kind, out) : eval_ref_variant<0, P64>(kind, out);
  }
  if (variant == 3) return eval_ref_variant<3, PMix>(kind, out);
  if (variant == 2) return eval_ref_variant<2, PMix>(kind, out);
  return variant ? eval_ref_variant<1, PMix>(kind, out) : eval_ref_variant<0, PMix>(kind, out);
}

static bool select_wide(uint32_t njobs) { return njobs <= kSelectWideJobs; }
KernelRef select_kernel_ref(uint32_t njobs) {
  if (select_wide(njobs)) return KernelRef{reinterpret_cast<const void *>(&k_select<1024>), 1024u, 1u};
  return KernelRef{reinterpret_cast<const void *>(&k_select<256>), 256u, 1u};
}
KernelRef zero_kernel_ref() { return KernelRef{reinterpret_cast<const void *>(&k_zero), 256u, 1u}; }

int eval_group_size(int kind, int variant) {
  const int d = kind_dim(kind);
  if (d == 1) return 0;   // 1-D integrals have no launch shapes (onedim.hip)
  const int k = d == 5 ? kNN1 : d == 6 ? kNN2 : kNN3;
  if (variant == 3) {
    return k == kNN1 ? KGroup<make_kv(kNN1, 3)>::G
                     : k == kNN2 ? KGroup<make_kv(kNN2, 3)>::G : KGroup<make_kv(kNN3, 3)>::G;
  }
  if (variant == 2) {
    return k == kNN1 ? KGroup<make_kv(kNN1, 2)>::G
                     : k == kNN2 ? KGroup<make_kv(kNN2, 2)>::G : KGroup<make_kv(kNN3, 2)>::G;
  }
  if (variant == 1) {
    return k == kNN1 ? KGroup<make_kv(kNN1, 1)>::G
                     : k == kNN2 ? KGroup<make_kv(kNN2, 1)>::G : KGroup<make_kv(kNN3, 1)>::G;
  }
  return k == kNN1 ? KGroup<kNN1>::G : k == kNN2 ? KGroup<kNN2>::G : KGroup<kNN3>::G;
}

hipError_t launch_roots(const RootsLaunch &L, hipStream_t s) {
  if (L.njobs == 0) return hipSuccess;
  hipLaunchKernelGGL(k_roots, dim3((L.njobs + 255) / 256), dim3(256), 0, s, L);
  return hipGetLastError();
}

hipError_t launch_select(const SelectLaunch &L, uint32_t njobs, hipStream_t s) {
  if (njobs == 0) return hipSuccess;
  if (select_wide(njobs)) hipLaunchKernelGGL((k_select<1024>), dim3(njobs), dim3(1024), 0, s, L);
  else hipLaunchKernelGGL((k_select<256>), dim3(njobs), dim3(256), 0, s, L);
  return hipGetLastError();
}

hipError_t launch_admit(const AdmitLaunch &L, hipStream_t s) {
  if (L.n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_admit, dim3((L.n + 255) / 256), dim3(256), 0, s, L);
  return hipGetLastError();
}

hipError_t launch_gather(const GatherLaunch &L, hipStream_t s) {
  if (L.n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather, dim3((L.n + 255) / 256), dim3(256), 0, s, L);
  return hipGetLastError();
}

hipError_t launch_zero(uint32_t *p, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_zero, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

}  // namespace g3l
