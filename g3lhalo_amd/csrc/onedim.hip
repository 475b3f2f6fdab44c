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
// Measured, a call to its results on the host: one HOD set (256 integrals)
// 3.7 -> 0.70 ms, 256 sets 104 -> 23 ms, the precomputation 118 -> 9.1 ms.  A round
// of a block is a chain of a few microseconds each: the selection of one wave,
// the scattered loads of the nodes' values (384 MB of nodes at 256 sets, 46 GB read from
// HBM), the rule's 450 dependent instructions, three barriers; two blocks per
// compute unit do not fill it.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "onedim.h"
#include "rules.h"
#include "select_math.h"
#include "select_wave.h"

#pragma clang fp contract(off)

namespace g3l {

namespace {

constexpr int kThreads = 512, kWaves = kThreads / 64;
static_assert(kWaves == kOneDimMaxUnit, "one wave per integral of a unit");
constexpr int kPts = 15, kRec = 16;
constexpr uint32_t kMaxSplit = kOneDimCap / 2;   // regions cut in one round
constexpr uint32_t kChunk = 32;                  // regions reduced together (precomputation)
static_assert(kChunk * kPts <= kThreads, "a point per thread");

// Device memory of a block: `nodes` nodes and the regions of `waves` integrals.
// A node's values lie together, in records of 16: a lane that reduces a node reads
// three cache lines where a row per point meant thirty, and the nodes of a wave's
// regions are neighbours only while the tree is young (one HOD set 0.77 -> 0.70 ms,
// 256 sets 25.2 -> 23.0).
struct Store {
  double2 *ab;            // [nodes][kRec]
  int32_t *ix;            // [nodes][kRec]
  double *c, *h;          // [nodes]
  double *val, *err;      // [waves][kOneDimCap]: rule value, error
  uint16_t *node;         // [waves][kOneDimCap]
  uint32_t nodes;
  __device__ __forceinline__ Store(unsigned char *p, uint32_t nodes_, uint32_t waves)
      : nodes(nodes_) {
    ab = reinterpret_cast<double2 *>(p);
    c = reinterpret_cast<double *>(ab + (size_t)kRec * nodes);
    h = c + nodes;
    val = h + nodes;
    err = val + (size_t)waves * kOneDimCap;
    ix = reinterpret_cast<int32_t *>(err + (size_t)waves * kOneDimCap);
    node = reinterpret_cast<uint16_t *>(ix + (size_t)kRec * nodes);
  }
};

// The nodes a block reads: the first nd of them, the whole top of the tree in
// breadth-first order, from its group's table (k_onedim_top; nd 0: none), the
// others from its own store.
struct TopStore {
  double2 ab[kOneDimTop][kRec];
  int32_t ix[kOneDimTop][kRec];
  double c[kOneDimTop], h[kOneDimTop];
};
struct Nodes {
  const TopStore *top;
  Store own;
  uint32_t nd;
  __device__ __forceinline__ double c(uint32_t id) const {
    return *(id < nd ? &top->c[id] : &own.c[id - nd]);
  }
  __device__ __forceinline__ double h(uint32_t id) const {
    return *(id < nd ? &top->h[id] : &own.h[id - nd]);
  }
};

struct WaveLds {
  SearchLds search;
  uint16_t split[kMaxSplit];   // slots of the batch, ascending
};

// The order of the arrays counts: with the nodes beside their slots, or the point
// values in the searches' memory, a 128-bin precomputation took 9.5 to 9.7 ms
// rather than 9.1.
struct Lds {
  WaveLds w[kWaves];
  // first of a node's two children, 0: none; of node id at id - the number of
  // nodes whose children are in the table (child_of)
  uint32_t child[kOneDimNodes];
  uint16_t fresh[kOneDimNodes / 2];    // nodes split for the first time this round
  double f[kChunk * kPts];             // point values (precomputation)
  uint32_t nnodes, nfresh, full;
  uint16_t n[kWaves], cut[kWaves];     // regions, and regions cut this round, per integral
  union {
    int32_t row[kWaves];               // n_bar: hmf row of each integral's redshift
    OneDimJob job[kWaves];             // precomputation: each integral's parameters
  };
  uint16_t node[kWaves][kMaxSplit];    // nodes of the batch, in its order
};
static_assert(2 * sizeof(Lds) <= 160 * 1024, "two blocks per compute unit");
// Dynamic LDS, so that the functions kept out of line address it as LDS.
extern __shared__ __align__(16) unsigned char lds_raw[];
__device__ __forceinline__ Lds &lds() { return *reinterpret_cast<Lds *>(lds_raw); }

// Nodes of the table whose children are in the table too.
__device__ __forceinline__ uint32_t inner(uint32_t nd) { return nd / 2; }
__device__ __forceinline__ uint32_t child_of(uint32_t nd, uint32_t v) {
  return v < inner(nd) ? 2 * v + 1 : lds().child[v - inner(nd)];
}

// The part of the integrand that depends on the abscissa alone.
//   n_bar: ab = (m, Ncen + Nsat), ix = the mass index;
//   sigma^2, d sigma^2/dm: ab = (amplitude T(k)^2, k^ns);
//   distance, amplitude: ab.x = the integrand (one integral per group).
//
// Out of line, like wave_round: the kernel's loops around the inlined code kept
// its FP64 constants in registers and spilled the rest (nbar of one HOD set
// 0.89 ms inlined, 0.77 so).
template <bool PRE>
__device__ __noinline__ void one_dim_node(const DevTables &T, const OneDimGroup &g, double t1,
                                             double x, double2 &ab, int32_t &ix) {
  if constexpr (!PRE) {
    TermArgs a{};
    a.h1 = g.h;
    a.rs1 = g.rs;
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
__device__ __noinline__ double precomp_point(int mode, const OneDimJob &j, double x,
                                                const double2 &ab) {
  if (mode == kOneDComoving || mode == kOneDAmplitude) return ab.x;
  const double spectrum = ab.x * j.t2 * j.t2 * ab.y;   // eh_spectrum's order
  const double W = tophat(x, j.t1);
  if (mode == kOneDSigma2) return x * x * W * W * spectrum;
  return x * x * W * d_tophat(x, j.t1) * j.t3 * spectrum;
}

// One integral's state; every field is the same in all lanes of its wave.
struct WaveState {
  uint32_t n, flags, K;
  double V;
};

// Totals, stop test and batch of one integral's n <= 64 R regions: its flags
// when it ends, otherwise the size K of the batch, whose slots are in W.split.
//
// The totals keep the order they have in k_select, whose 256 threads take the
// slots in strides and then add pairwise: lane l holds the threads l, l + 64,
// l + 128 and l + 192.
template <int R>
__device__ __noinline__ WaveState wave_round(const double *val, const double *err, double reltol,
                                             uint32_t n) {
  const int lane = threadIdx.x & 63;
  WaveLds &W = lds().w[threadIdx.x >> 6];
  WaveState st{n, 0, 0, 0.0};
  constexpr int V4 = R < 4 ? R : 4;
  constexpr int B = R < 8 ? R : 8;   // loads in flight per array
  uint64_t k[R];
  double vs[V4] = {}, vc[V4] = {}, es[V4] = {};
  double check = 0;   // NaN once a value or error is not finite
  uint64_t maxkey = 0;
#pragma unroll
  for (int r0 = 0; r0 < R; r0 += B) {
    if (64u * r0 >= n) {
#pragma unroll
      for (int r = 0; r < B; ++r) k[r0 + r] = ~0ull;
      continue;
    }
    double v[B], e[B];
#pragma unroll
    for (int r = 0; r < B; ++r) {
      const uint32_t i = 64 * (r0 + r) + lane;
      v[r] = i < n ? val[i] : 0.0;
      e[r] = i < n ? err[i] : 0.0;
    }
#pragma unroll
    for (int r = 0; r < B; ++r) {
      check = fma(0.0, v[r], fma(0.0, e[r], check));
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
      vc[q] += vc[q + w] + sum_error(a, b, t);
      vs[q] = t;
      es[q] += es[q + w];
    }
  }
  const double V = comp_total(vs[0], vc[0]);
  double E = es[0];
  tree([&](auto w) { E += from_above<decltype(w)::value>(E); });
  E = readlane64(E, 0);
  st.V = V;
  st.K = 0;
  if (__ballot(check != check) != 0) st.flags |= kJobNonfinite;
  const double thr = fabs(V) * reltol;
  if (!(E > 0 && E > thr)) {
    st.flags |= kJobDone | kJobConverged;
    return st;
  }
  // every key is among these, so the boundary is
  Boundary Bd{};
  (void)find_boundary<R>(k, n, wave_max(maxkey), Goal{thr, ~0ull, 0, 0.0}, W.search, Bd);
  const uint32_t K = Bd.gt + Bd.take;
  if (n + K > kOneDimCap) {
    st.flags |= kJobDone | kJobPoolFull;
    return st;
  }
  st.K = K;
  // regions above T and the first `take` of those at T, in slot order
  uint32_t at = 0, ties = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (64u * r >= n) break;
    const bool in = k[r] != ~0ull;
    bool s = in && k[r] >= Bd.T;
    if (Bd.take != Bd.eq) {
      const bool tie = in && k[r] == Bd.T;
      const uint64_t tm = __ballot(tie);
      s = s && (!tie || ties + lanes_below(tm) < Bd.take);
      ties += (uint32_t)__popcll(tm);
    }
    const uint64_t sm = __ballot(s);
    if (s) W.split[at + lanes_below(sm)] = (uint16_t)(64 * r + lane);
    at += (uint32_t)__popcll(sm);
  }
  return st;
}

// One round of this wave's integral, by the number of its regions, and the
// nodes its batch needs: the first wave to split a node makes its children.
__device__ __forceinline__ void wave_select(const double *val, const double *err,
                                            const uint16_t *node, double reltol, uint32_t nd,
                                            uint32_t limit, WaveState &st) {
  if (st.n <= 64) st = wave_round<1>(val, err, reltol, st.n);
  else if (st.n <= 256) st = wave_round<4>(val, err, reltol, st.n);
  else if (st.n <= 1024) st = wave_round<16>(val, err, reltol, st.n);
  else st = wave_round<32>(val, err, reltol, st.n);
  Lds &S = lds();
  const WaveLds &W = S.w[threadIdx.x >> 6];
  wave_sync();
  for (uint32_t a = threadIdx.x & 63; a < st.K; a += 64) {
    const uint32_t v = node[W.split[a]];
    S.node[threadIdx.x >> 6][a] = (uint16_t)v;
    if (v < inner(nd)) continue;
    uint32_t *child = S.child - inner(nd);
    if (atomicCAS(&child[v], 0u, ~0u) == 0u) {
      const uint32_t id = atomicAdd(&S.nnodes, 2u);
      if (id + 2 <= limit) {
        child[id] = 0;
        child[id + 1] = 0;
        child[v] = id;
        S.fresh[atomicAdd(&S.nfresh, 1u)] = (uint16_t)v;
      } else {
        child[v] = 0;
        S.full = 1;
      }
    }
  }
}

// Region i of the block's round: region r = i / count of integral w = i mod
// count (false if it has fewer), its node and its slot.  An integral's regions
// are the left (even) and right (odd) halves of those in its W.split; the left
// half keeps its parent's slot, the right one takes the next free slot.  The
// parent's node comes from S.node: its slot's entry in memory is the left half's
// from the moment that is reduced, which may be before another wave, a later
// chunk or a later pass of this one comes to the right half.
// Neighbouring lanes take the same rank of different integrals, mostly the
// same node, whose values they then read together.
__device__ __forceinline__ bool place(const Nodes &N, uint32_t i, uint32_t count, bool root,
                                      uint32_t &w, uint32_t &id, uint32_t &slot) {
  const Lds &S = lds();
  const uint32_t r = i / count;
  w = i - r * count;
  id = 0;
  slot = 0;
  if (root) return true;
  if (r >= 2 * S.cut[w]) return false;
  id = child_of(N.nd, S.node[w][r >> 1]) + (r & 1u);
  slot = (r & 1u) ? S.n[w] + (r >> 1) : S.w[w].split[r >> 1];
  return true;
}

// gk_reduce out of line.
__device__ __noinline__ double2 gk_sums(const double *f, double h) {
  double2 r;
  gk_reduce(f, h, r.x, r.y);
  return r;
}

// Rule sums of the `total` regions (place) of the round of the block's `count`
// integrals, or of their roots.  Every thread of the block calls it.
template <bool PRE>
__device__ __forceinline__ void block_reduce(const OneDimLaunch &L, int mode, const Nodes &N,
                                             uint32_t count, uint32_t total, bool root) {
  Lds &S = lds();
  const Store &G = N.own;
  const uint32_t tid = threadIdx.x;
  if constexpr (!PRE) {
    // a region per thread: a point is two loads, a table look-up and two products
    for (uint32_t i = tid; i < total; i += kThreads) {
      uint32_t w, id, slot;
      if (!place(N, i, count, root, w, id, slot)) continue;
      const double *hmf = L.T.hmf + S.row[w];
      const bool top = id < N.nd;
      const double2 *ab = top ? N.top->ab[id] : G.ab + (size_t)(id - N.nd) * kRec;
      const int32_t *ix = top ? N.top->ix[id] : G.ix + (size_t)(id - N.nd) * kRec;
      double f[kPts], v, e;
#pragma unroll
      for (int j = 0; j < kPts; ++j) {
        const double2 q = ab[j];
        f[j] = q.x * hmf[ix[j]] * q.y;
      }
      gk_reduce(f, N.h(id), v, e);
      G.val[w * kOneDimCap + slot] = v;
      G.err[w * kOneDimCap + slot] = e;
      G.node[w * kOneDimCap + slot] = (uint16_t)id;
    }
  } else {
    // a point per thread: a point takes the window's sin and cos of a large
    // argument, and in most rounds every integral has two regions
    for (uint32_t i0 = 0; i0 < total; i0 += kChunk) {
      const uint32_t q = tid / kPts, i = i0 + q, j = tid - kPts * q;
      uint32_t w, id, slot;
      if (q < kChunk && i < total && place(N, i, count, root, w, id, slot)) {
        const double c = N.c(id), h = N.h(id);
        double x;
        rule_point<1>((int)j, &c, &h, &x);
        S.f[tid] = precomp_point(mode, S.job[w], x, G.ab[(size_t)id * kRec + j]);
      }
      __syncthreads();
      if (tid < kChunk && i0 + tid < total && place(N, i0 + tid, count, root, w, id, slot)) {
        const double2 r = gk_sums(S.f + kPts * tid, N.h(id));
        G.val[w * kOneDimCap + slot] = r.x;
        G.err[w * kOneDimCap + slot] = r.y;
        G.node[w * kOneDimCap + slot] = (uint16_t)id;
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
  const Store G(L.store + (size_t)blockIdx.x * L.store_bytes, L.nodes, L.waves);
  Nodes N{nullptr, G, PRE ? 0u : L.top ? kOneDimTop : 0u};
  const uint32_t in = inner(N.nd);
  // ids end where the children's table or the store does
  const uint32_t limit = min(in + kOneDimNodes, N.nd + L.nodes);
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
    const bool reuse = have == U.group && S.nnodes - N.nd <= L.nodes / 2;
    if (N.nd) N.top = reinterpret_cast<const TopStore *>(L.top) + U.group;
    const double t1 = L.jobs[g.job0 + U.first].t1;
    if (tid < (int)U.count) {
      const OneDimJob job = L.jobs[g.job0 + U.first + tid];
      if constexpr (PRE) S.job[tid] = job;
      else S.row[tid] = zix_round(L.T, job.t1) * L.T.nb;
    }
    __syncthreads();
    if (!reuse) {
      if (N.nd) {   // the table's last level has no children yet
        if (tid == 0) S.nnodes = N.nd;
        for (uint32_t v = tid; v < N.nd - in; v += kThreads) S.child[v] = 0;
      } else {
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
          one_dim_node<PRE>(L.T, g, t1, x, G.ab[tid], G.ix[tid]);
        }
      }
    }
    if (tid == 0) S.full = 0;
    __syncthreads();
    WaveState st{1, mine ? 0u : (uint32_t)kJobDone, 0, 0.0};
    block_reduce<PRE>(L, g.mode, N, U.count, U.count, true);
    bool again = false;
    for (;;) {
      if (tid == 0) S.nfresh = 0;
      __syncthreads();
      st.K = 0;
      if (!(st.flags & kJobDone)) {
        const size_t at = (size_t)wave * kOneDimCap;
        wave_select(G.val + at, G.err + at, G.node + at, L.reltol, N.nd, limit, st);
      }
      if (lane == 0) {
        S.n[wave] = (uint16_t)st.n;
        S.cut[wave] = (uint16_t)st.K;
      }
      __syncthreads();
      uint32_t most = 0;
#pragma unroll
      for (int q = 0; q < kWaves; ++q) most = S.cut[q] > most ? S.cut[q] : most;
      const uint32_t total = 2 * most * U.count;
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
        const uint32_t v = S.fresh[pr], id = S.child[v - in] + right - N.nd;
        // the halves of a split, as in the cut of src/hcubature.cpp:206-218
        const double h = N.h(v) * 0.5, c = right ? N.c(v) + h : N.c(v) - h;
        double x;
        rule_point<1>(j, &c, &h, &x);
        one_dim_node<PRE>(L.T, g, t1, x, G.ab[(size_t)id * kRec + j], G.ix[(size_t)id * kRec + j]);
        if (j == 0) {
          G.c[id] = c;
          G.h[id] = h;
        }
      }
      if (np) __syncthreads();
      block_reduce<PRE>(L, g.mode, N, U.count, total, false);
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

// The top of every group's tree, kOneDimTop nodes in breadth-first order, a
// point per thread (n_bar).  With fewer than two groups for every resident
// block, several blocks would evaluate the same nodes, and a block alone with
// one integral spends most of its time on them.
__global__ __launch_bounds__(256) void k_onedim_top(OneDimLaunch L, TopStore *top) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kOneDimTop * kPts) return;
  const int j = (int)(i / kOneDimTop);
  const uint32_t id = i - (uint32_t)j * kOneDimTop;
  const OneDimGroup &g = L.groups[blockIdx.y];
  // the path from the root: the bits of id + 1 below its leading one
  double c = 0.5 * (g.lo + g.hi), h = 0.5 * (g.hi - g.lo), x;
  for (int b = 30 - __clz((int)(id + 1)); b >= 0; --b) {
    h *= 0.5;
    c = (id + 1) >> b & 1u ? c + h : c - h;
  }
  rule_point<1>(j, &c, &h, &x);
  TopStore &t = top[blockIdx.y];
  one_dim_node<false>(L.T, g, 0.0, x, t.ab[id][j], t.ix[id][j]);
  if (j == 0) {
    t.c[id] = c;
    t.h[id] = h;
  }
}

size_t one_dim_store_bytes(uint32_t nodes, uint32_t waves) {
  const size_t b = (size_t)nodes * (kRec * (sizeof(double2) + sizeof(int32_t)) + 2 * sizeof(double)) +
                   (size_t)waves * kOneDimCap * (2 * sizeof(double) + sizeof(uint16_t));
  return (b + 255) / 256 * 256;
}
size_t one_dim_top_bytes() { return sizeof(TopStore); }
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

hipError_t launch_one_dim_top(const OneDimLaunch &L, uint32_t ngroups, hipStream_t s) {
  if (ngroups == 0 || ngroups > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_onedim_top, dim3((kOneDimTop * kPts + 255) / 256, ngroups), dim3(256), 0, s, L,
                     reinterpret_cast<TopStore *>(L.top));
  return hipGetLastError();
}

hipError_t launch_one_dim(bool precomp, const OneDimLaunch &L, uint32_t blocks, hipStream_t s) {
  if (L.nunits == 0) return hipSuccess;
  if (blocks == 0 || blocks > L.nunits || (precomp && L.top) || L.nodes == 0 ||
      L.nodes > kOneDimNodes || L.waves == 0 || L.waves > (uint32_t)kOneDimMaxUnit ||
      L.store_bytes < one_dim_store_bytes(L.nodes, L.waves))
    return hipErrorInvalidValue;
  return precomp ? launch<true>(L, blocks, s) : launch<false>(L, blocks, s);
}

}  // namespace g3l
