// engine.cpp -- host side of the gfx950 NNMap / NMapMap engine: context and
// tables in HBM, HOD sets with device n_bar(z), the plain host-driven
// cubature and the device-resident batched cubature, behind the C ABI of
// include/g3l.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <new>
#include <vector>

#include "engine.h"

using namespace g3l;

namespace {

// Constants of the reference (src/constants.h:15-39, src/Cosmology.h:27-28).
const double kPi = 3.14159;
const double kLn10 = std::log(10.0);
const double kC = 2.99792e5;
const double kGMsun = 1.327e11;
const double kMpcKm = 3.086e19;

// A sigma below 1e-300 is as good as 1e-300: log(m / M_th) is zero or at least
// 1e-16, so the error function saturates either way, and x / sigma stays finite.
DevHod to_dev(const g3l_hod &h) {
  return DevHod{h.f, h.alpha, h.mth, std::max(h.sigma, 1e-300), h.mprime, h.beta};
}

}  // namespace

namespace g3l {

int kind_of(int stat, int term) { return stat == G3L_NNMAP ? term : 3 + term; }

KindLaunch kind_launch(const g3l_ctx *c, int prec) {
  KindLaunch L;
  for (int k = 0; k < kNumKinds; ++k) {
    const bool mixed = prec == G3L_MIXED && (c->mixed_fp32_kinds >> k & 1u);
    L.prec[k] = mixed ? G3L_MIXED : G3L_FP64;
    L.variant[k] = c->variant[mixed][k];
  }
  return L;
}

const double *nbar_ptr(const g3l_ctx *c, int set, int which) {
  return c->nbar_chunks[set / kSetsPerChunk].dev.as<double>() +
         ((size_t)(set % kSetsPerChunk) * 2 + which) * c->nb;
}

// Log-space HOD constants: log(mmin/M_th), log(mmin/M'), log(mmin).
void fill_logs(const g3l_ctx *c, TermArgs &a) {
  a.lmmin = std::log(c->mmin);
  a.lth1 = std::log(c->mmin / a.h1.mth);
  a.lmp1 = std::log(c->mmin / a.h1.mprime);
  a.lth2 = std::log(c->mmin / a.h2.mth);
  a.lmp2 = std::log(c->mmin / a.h2.mprime);
}

// HOD and n_bar selection by type (src/NNMap_Model.cu:437-475); NMapMap uses
// its one HOD (slot 1).
TermArgs make_args(const g3l_ctx *c, const g3l_request &r) {
  const HodSet &s = c->sets[r.hodset];
  TermArgs a{};
  a.t1 = r.theta[0];
  a.t2 = r.theta[1];
  a.t3 = r.theta[2];
  a.A = s.A;
  a.eps = s.eps;
  if (r.stat == G3L_NMAPMAP) {
    a.h1 = a.h2 = to_dev(s.h1);
    a.nb1 = a.nb2 = nbar_ptr(c, r.hodset, 0);
    a.same = 1;
  } else {
    bool a1 = r.type1 == 1, a2 = r.type2 == 1;
    a.h1 = to_dev(a1 ? s.h1 : s.h2);
    a.nb1 = nbar_ptr(c, r.hodset, a1 ? 0 : 1);
    a.h2 = to_dev(a2 ? s.h1 : s.h2);
    a.nb2 = nbar_ptr(c, r.hodset, a2 ? 0 : 1);
    a.same = (a1 == a2) || s.identical;
  }
  a.rs1 = 1. / a.h1.sigma;
  a.rs2 = 1. / a.h2.sigma;
  fill_logs(c, a);
  return a;
}

// Integration box of a term (src/NNMap_Model.cu:313-314, 338-339, 363-364).
int term_box(const g3l_ctx *c, int term, double *lo, double *hi) {
  int d = 0;
  lo[d] = std::log10(0.1);
  hi[d++] = std::log10(1e6);
  lo[d] = std::log10(0.1);
  hi[d++] = std::log10(1e6);
  lo[d] = 0;
  hi[d++] = 2 * kPi;
  for (int i = 0; i < term; ++i) {
    lo[d] = std::log10(c->mmin_i);
    hi[d++] = std::log10(c->mmax_i);
  }
  lo[d] = c->zmin_i;
  hi[d++] = c->zmax_i;
  return d;
}

// Prefactors (src/NNMap_Model.cu:321-322, 346-347, 371-372;
// src/NMapMap_Model.cu:188-190, 212-214, 235-237).
double prefactor(const g3l_ctx *c, int stat, int term, double r) {
  const double tp = 2 * kPi;
  double v;
  if (stat == G3L_NNMAP) v = r * 3 * c->H0 * c->H0 * c->Om / 2 / kC / kC;
  else v = r * 9 * std::pow(c->H0, 4) * std::pow(c->Om, 2) / 4 / std::pow(kC, 4);
  for (int i = 0; i < 2 + term; ++i) v = v * kLn10;
  return v / tp / tp / tp;
}

int check_request(const g3l_ctx *c, const g3l_request &r) {
  if (r.stat != G3L_NNMAP && r.stat != G3L_NMAPMAP) return G3L_EINVAL;
  if (r.term < 1 || r.term > 3) return G3L_EINVAL;
  if (r.hodset < 0 || r.hodset >= (int)c->sets.size()) return G3L_EINVAL;
  if (!(r.reltol >= 0) || !std::isfinite(r.theta[0]) || !std::isfinite(r.theta[1]) ||
      !std::isfinite(r.theta[2]))
    return G3L_EINVAL;
  return G3L_OK;
}

int status_of(uint32_t flags) {
  if (flags & kJobPoolFull) return G3L_ENOMEM_POOL;
  if (flags & kJobNonfinite) return G3L_NONFINITE;
  if (flags & kJobCapped) return G3L_MAXEVAL_HIT;
  return G3L_OK;
}

// Slot capacity of one integral: with a budget, the last pop happens while
// numEval < maxEval, so n <= 1 + (maxEval + pts) / (2 pts).
uint32_t slot_cap(uint64_t maxeval, int pts, uint32_t unlimited_cap) {
  if (maxeval == 0) return unlimited_cap;
  uint64_t c = 2 + (maxeval + (uint64_t)pts) / (2ull * (uint64_t)pts);
  return (uint32_t)std::min<uint64_t>(c, 1ull << 26);
}

}  // namespace g3l

namespace g3l {

int ctx_create_bare(g3l_ctx **out) {
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return G3L_ENODEV;
  g3l_ctx *c = new (std::nothrow) g3l_ctx();
  if (!c) return G3L_ENOMEM;
  if (hipGetDevice(&c->device) != hipSuccess ||
      hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return G3L_EHIP;
  }
  bool ok = true;
  for (auto &e : c->ev) ok = ok && hipEventCreate(&e) == hipSuccess;
  for (auto &e : c->kev) ok = ok && hipEventCreate(&e) == hipSuccess;
  if (!ok) {
    g3l_ctx_destroy(c);
    return G3L_EHIP;
  }
  // the allocation-free entry point's array on this device (a failure is
  // reported here and again by that entry point, which retries)
  (void)scratch_resolve(c->device);
  *out = c;
  return G3L_OK;
}

// ---------------------------------------------------------------------------
// Batched engine: all jobs refine together; per round one selection launch
// and one evaluation launch per integrand kind, or one for all kinds while a
// round is small.

// Rounds queued at a time at most, and most blocks of a round that is queued
// before the last one's outcome is known (its blocks are a bound, mostly twice
// what it needs; anything from 512 to 20000 takes the same time).
constexpr uint32_t kBurstRounds = 16;
constexpr uint64_t kBurstBlocks = 4096;

int refine_jobs(g3l_ctx *c, const EngineBufs &B, uint32_t nj, bool timed, int prec,
                bool use_graph) {
  hipStream_t s = c->stream;
  uint32_t *dcnt = B.dcnt;
  uint32_t *hcnt = B.hcnt;
  EvalItem *lists[kNumKinds];
  for (int k = 0; k < kNumKinds; ++k) lists[k] = B.lists[k];
  const uint64_t *per_kind = B.per_kind;
  const uint64_t slots = B.slots;
  int rc;

  RootsLaunch R{};
  R.jobs = B.jobs;
  R.boxes = B.boxes;
  R.state = B.state;
  R.geo = B.geo;
  R.split = B.split;
  R.stride = slots;
  for (int k = 0; k < kNumKinds; ++k) R.lists[k] = lists[k];
  R.counters = dcnt;
  R.njobs = nj;
  G3L_HIP(launch_zero(dcnt, kNumKinds + 1, s));
  if (B.rows) G3L_HIP(launch_zero(B.rows, kRows * kRowWords, s));
  G3L_HIP(launch_roots(R, s));

  EvalLaunch EL{};
  EL.T = c->T;
  EL.args = B.args;
  EL.jobs = B.jobs;
  EL.geo = B.geo;
  EL.split = B.split;
  EL.stride = slots;
  EL.njobs = nj;

  SelectLaunch SL{};
  SL.jobs = B.jobs;
  SL.state = B.state;
  SL.geo = B.geo;
  SL.split = B.split;
  SL.stride = slots;
  for (int k = 0; k < kNumKinds; ++k) {
    SL.lists[k] = lists[k];
    SL.list_cap[k] = (uint32_t)std::min<uint64_t>(per_kind[k], 0xffffffffull);
  }
  SL.counters = dcnt;
  SL.trace = B.trace;
  SL.trace_cap = B.trace ? B.trace_cap : 0;

  double eval_ms = 0, select_ms = 0;
  double kind_ms[kNumKinds] = {0};
  uint64_t kind_launches[kNumKinds] = {0};
  bool kind_used[kNumKinds];
  uint64_t launches = 0;
  uint32_t rounds = 0;
  // the roots' lists: an entry per integral
  for (int k = 0; k < kNumKinds; ++k) hcnt[k] = B.kind_jobs[k];
  // regions of each kind, a bound (finished integrals' count too): a round's list
  // has at most two entries for each
  uint64_t live[kNumKinds];
  for (int k = 0; k < kNumKinds; ++k) live[k] = B.kind_jobs[k];
  // graph mode: the round's launches and the counter copy are one graph
  // (every node records its events; they are read only when timed)
  RoundGraph &graph = c->graph;
  const KindLaunch KL = kind_launch(c, prec);
  auto ready_graph = [&]() -> int {
    // the executable graph is kept while the kinds, variants, precision,
    // job count and buffers stay the same (repeated calls of one workload)
    bool in_run[kNumKinds];
    std::vector<uint64_t> key = {nj, slots, (uint64_t)(uintptr_t)B.geo,
                                 (uint64_t)(uintptr_t)lists[0], (uint64_t)(uintptr_t)B.jobs,
                                 (uint64_t)(uintptr_t)B.state, (uint64_t)(uintptr_t)B.args,
                                 (uint64_t)(uintptr_t)B.split, (uint64_t)(uintptr_t)dcnt,
                                 (uint64_t)(uintptr_t)hcnt, (uint64_t)(uintptr_t)SL.trace,
                                 SL.trace_cap};
    for (int k = 0; k < kNumKinds; ++k) {
      in_run[k] = per_kind[k] != 0;
      key.push_back(per_kind[k]);
      key.push_back((uint64_t)KL.prec[k]);
      key.push_back((uint64_t)KL.variant[k]);
    }
    if (!graph.exec || key != c->graph_key) {
      c->graph_key.clear();
      if ((rc = graph.build(in_run, KL.prec, KL.variant, EL, SL, dcnt, kNumKinds + 1, hcnt, c->ev,
                            c->kev, nj)))
        return rc;
      c->graph_key = key;
    }
    return G3L_OK;
  };
  // Small rounds: every kind's evaluation in one launch, and rounds queued
  // without waiting for the last one while the bound on their blocks stays
  // small.  FP64 kinds only.
  bool small_ok = B.rows != nullptr;
  for (int k = 0; k < kNumKinds; ++k) small_ok = small_ok && (!per_kind[k] || KL.prec[k] == G3L_FP64);
  uint32_t row = 0;
  int clock_khz = 0;
  if (small_ok && timed)
    G3L_HIP(hipDeviceGetAttribute(&clock_khz, hipDeviceAttributeWallClockRate, c->device));
  // the rounds from the lists of length hcnt on; the last one's counters to hcnt
  auto run_small = [&]() -> int {
    uint64_t bound[kNumKinds], most[kNumKinds];
    for (int k = 0; k < kNumKinds; ++k) {
      bound[k] = std::min<uint64_t>(hcnt[k], per_kind[k]);
      most[k] = live[k];
    }
    if (row + kBurstRounds + 1 > kRows) {
      G3L_HIP(launch_zero(B.rows, kRows * kRowWords, s));
      row = 0;
    }
    const uint32_t first = row;
    EvalSmallLaunch ES{};
    ES.E = EL;
    for (int k = 0; k < kNumKinds; ++k) {
      ES.lists[k] = lists[k];
      ES.count[k] = (uint32_t)bound[k];
    }
    uint32_t n = 0;
    do {
      small_ends(bound, ES.end);
      uint32_t *here = B.rows + (size_t)row * kRowWords;
      ES.row = n ? here - kRowWords : nullptr;
      ES.clock = reinterpret_cast<uint64_t *>(here);
      G3L_HIP(launch_eval_small(ES, s));
      SelectLaunch SR = SL;
      SR.counters = here;
      SR.clock = ES.clock;
      G3L_HIP(launch_select(SR, nj, s));
      ++row;
      ++n;
      for (int k = 0; k < kNumKinds; ++k) {
        bound[k] = std::min<uint64_t>(2 * most[k], per_kind[k]);
        most[k] *= 2;
      }
    } while (n < kBurstRounds && small_blocks(bound) <= kBurstBlocks);
    G3L_HIP(hipMemcpyAsync(B.hrows, B.rows + (size_t)first * kRowWords,
                           (size_t)n * kRowWords * sizeof(uint32_t), hipMemcpyDeviceToHost, s));
    G3L_HIP(hipStreamSynchronize(s));
    for (uint32_t r = 0; r < n; ++r) {
      const uint32_t *h = B.hrows + (size_t)r * kRowWords;
      const uint64_t *t = reinterpret_cast<const uint64_t *>(h);
      uint64_t eval_end = t[kRowStart];
      for (int k = 1; k < kNumKinds; ++k) {
        if (!hcnt[k]) continue;
        ++launches;
        ++kind_launches[k];
        if (!clock_khz) continue;
        eval_end = std::max(eval_end, t[kRowKindEnd + k]);
        kind_ms[k] += (double)(t[kRowKindEnd + k] - t[kRowStart]) / clock_khz;
      }
      if (clock_khz) {
        eval_ms += (double)(eval_end - t[kRowStart]) / clock_khz;
        if (t[kRowSelectEnd] > t[kRowSelect])
          select_ms += (double)(t[kRowSelectEnd] - t[kRowSelect]) / clock_khz;
      }
      for (int k = 0; k <= kNumKinds; ++k) hcnt[k] = h[k];
      for (int k = 0; k < kNumKinds; ++k) live[k] += hcnt[k] / 2;
      ++rounds;
      if (hcnt[kNumKinds] == 0) break;
    }
    return G3L_OK;
  };
  bool have_graph = false;
  for (;;) {
    if (small_ok) {
      uint64_t now[kNumKinds];
      for (int k = 0; k < kNumKinds; ++k) now[k] = hcnt[k];
      if (small_blocks(now) <= kSmallBlocks) {
        if ((rc = run_small())) return rc;
        if (hcnt[kNumKinds] == 0) break;
        continue;
      }
    }
    if (use_graph && !have_graph) {
      if ((rc = ready_graph())) return rc;
      have_graph = true;
    }
    uint32_t cnt[kNumKinds];
    for (int k = 0; k < kNumKinds; ++k) {
      cnt[k] = (uint32_t)std::min<uint64_t>(hcnt[k], per_kind[k]);
      kind_used[k] = cnt[k] != 0;
      if (!kind_used[k]) continue;
      ++launches;
      ++kind_launches[k];
    }
    if (use_graph) {
      if ((rc = graph.launch(cnt, lists, nj, s))) return rc;
    } else {
      if (timed) G3L_HIP(hipEventRecord(c->ev[0], s));
      for (int k = 0; k < kNumKinds; ++k) {
        if (!kind_used[k]) continue;
        EL.list = lists[k];
        EL.count = cnt[k];
        if (timed) G3L_HIP(hipEventRecord(c->kev[2 * k], s));
        G3L_HIP(launch_eval(k, KL.prec[k], KL.variant[k], EL, s));
        if (timed) G3L_HIP(hipEventRecord(c->kev[2 * k + 1], s));
      }
      if (timed) G3L_HIP(hipEventRecord(c->ev[1], s));
      G3L_HIP(launch_zero(dcnt, kNumKinds + 1, s));
      G3L_HIP(launch_select(SL, nj, s));
      if (timed) G3L_HIP(hipEventRecord(c->ev[2], s));
      G3L_HIP(hipMemcpyAsync(hcnt, dcnt, (kNumKinds + 1) * sizeof(uint32_t), hipMemcpyDeviceToHost,
                             s));
    }
    G3L_HIP(hipStreamSynchronize(s));
    if (timed) {
      float a = 0, b = 0;
      G3L_HIP(hipEventElapsedTime(&a, c->ev[0], c->ev[1]));
      G3L_HIP(hipEventElapsedTime(&b, c->ev[1], c->ev[2]));
      eval_ms += a;
      select_ms += b;
      for (int k = 0; k < kNumKinds; ++k) {
        if (!kind_used[k]) continue;
        float m = 0;
        G3L_HIP(hipEventElapsedTime(&m, c->kev[2 * k], c->kev[2 * k + 1]));
        kind_ms[k] += m;
      }
    }
    ++rounds;
    for (int k = 0; k < kNumKinds; ++k) live[k] += hcnt[k] / 2;
    if (hcnt[kNumKinds] == 0) break;
  }
  c->last.eval_ms = eval_ms;
  c->last.select_ms = select_ms;
  c->last.eval_launches = launches;
  c->last.rounds = rounds;
  for (int k = 0; k < 8; ++k) {
    c->last.kind_ms[k] = k < kNumKinds ? kind_ms[k] : 0;
    c->last.kind_launches[k] = k < kNumKinds ? kind_launches[k] : 0;
  }
  return G3L_OK;
}

void finish_stats(g3l_ctx *c, const JobDesc *desc, const JobState *st, uint32_t nj,
                  double wall_ms) {
  uint64_t evals = 0;
  uint64_t kind_evals[kNumKinds] = {0};
  for (uint32_t j = 0; j < nj; ++j) {
    evals += st[j].neval;
    kind_evals[desc[j].kind] += st[j].neval;
  }
  c->last.wall_ms = wall_ms;
  c->last.evals = evals;
  for (int k = 0; k < 8; ++k) c->last.kind_evals[k] = k < kNumKinds ? kind_evals[k] : 0;
}

int run_engine(g3l_ctx *c, EngineJobs &E, std::vector<JobState> &out, bool timed, int prec,
               bool trace) {
  const uint32_t nj = (uint32_t)E.desc.size();
  out.assign(nj, JobState{});
  if (nj == 0) return G3L_OK;
  auto t0 = std::chrono::steady_clock::now();
  EngineBufs B{};
  for (auto &d : E.desc) {
    d.base = (uint32_t)B.slots;
    B.slots += d.cap;
    B.per_kind[d.kind] += 2ull * d.cap;
    ++B.kind_jobs[d.kind];
  }
  if (B.slots >= (1ull << 32) - 1) return G3L_ENOMEM;
  uint64_t list_total = 0;
  for (int k = 0; k < kNumKinds; ++k) list_total += B.per_kind[k];
  int rc;
  if ((rc = c->pool.ensure(B.slots * kNumFields * sizeof(double)))) return rc;
  if ((rc = c->split.ensure(B.slots))) return rc;
  if ((rc = c->lists.ensure(list_total * sizeof(EvalItem)))) return rc;
  if ((rc = c->jobs.ensure(nj * sizeof(JobDesc)))) return rc;
  if ((rc = c->state.ensure(nj * sizeof(JobState)))) return rc;
  if ((rc = c->args.ensure(E.args.size() * sizeof(TermArgs)))) return rc;
  if ((rc = c->boxes.ensure(E.boxes.size() * sizeof(double)))) return rc;
  // the counters, and behind them the rows
  constexpr size_t kCountBytes = 64 + kRows * kRowWords * sizeof(uint32_t);
  if ((rc = c->counters.ensure(kCountBytes))) return rc;
  if ((rc = c->hcounters.ensure(kCountBytes))) return rc;
  hipStream_t s = c->stream;
  if (trace && c->trace_cap > 0) {
    const size_t entries = (size_t)nj * c->trace_cap;
    if (entries > 0x7fffffffull) return G3L_EINVAL;
    if ((rc = c->trace.ensure(entries * sizeof(uint32_t)))) return rc;
    G3L_HIP(launch_zero(c->trace.as<uint32_t>(), (int)entries, s));
    B.trace = c->trace.as<uint32_t>();
    B.trace_cap = c->trace_cap;
  }
  G3L_HIP(hipMemcpyAsync(c->jobs.p, E.desc.data(), nj * sizeof(JobDesc), hipMemcpyHostToDevice, s));
  G3L_HIP(hipMemcpyAsync(c->args.p, E.args.data(), E.args.size() * sizeof(TermArgs),
                         hipMemcpyHostToDevice, s));
  G3L_HIP(hipMemcpyAsync(c->boxes.p, E.boxes.data(), E.boxes.size() * sizeof(double),
                         hipMemcpyHostToDevice, s));
  {
    uint64_t off = 0;
    for (int k = 0; k < kNumKinds; ++k) {
      B.lists[k] = c->lists.as<EvalItem>() + off;
      off += B.per_kind[k];
    }
  }
  B.geo = c->pool.as<double>();
  B.split = c->split.as<uint8_t>();
  B.jobs = c->jobs.as<JobDesc>();
  B.state = c->state.as<JobState>();
  B.args = c->args.as<TermArgs>();
  B.boxes = c->boxes.as<double>();
  B.dcnt = c->counters.as<uint32_t>();
  B.hcnt = c->hcounters.as<uint32_t>();
  B.rows = B.dcnt + 16;
  B.hrows = B.hcnt + 16;
  if ((rc = refine_jobs(c, B, nj, timed, prec, c->launch_mode == G3L_LAUNCH_GRAPH))) return rc;
  G3L_HIP(hipMemcpyAsync(out.data(), B.state, nj * sizeof(JobState), hipMemcpyDeviceToHost, s));
  G3L_HIP(hipStreamSynchronize(s));
  if (B.trace) {
    c->trace_jobs = nj;
    c->trace_rounds.resize(nj);
    for (uint32_t j = 0; j < nj; ++j) c->trace_rounds[j] = out[j].rounds;
  }
  auto t1 = std::chrono::steady_clock::now();
  finish_stats(c, E.desc.data(), out.data(), nj,
               std::chrono::duration<double, std::milli>(t1 - t0).count());
  return G3L_OK;
}

// ---------------------------------------------------------------------------
// 1-D integrals (k_onedim).

// Most integrals of a launch: group and integral numbers have to fit the kernel's words,
// and its lists grow with them.  Every resident block still has a hundred units and
// more, so that what the last ones take alone is small.
constexpr size_t kOneDimBatch = 1u << 20;

static int run_one_dim_batch(g3l_ctx *c, const std::vector<OneDimGroup> &groups,
                             const std::vector<OneDimJob> &jobs, bool precomp, double reltol,
                             double scale) {
  int cus = 0;
  G3L_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
  size_t total = 0;
  for (const OneDimGroup &g : groups) total += g.count;
  if (groups.size() > kOneDimBatch || total > kOneDimBatch) return G3L_EINVAL;
  const size_t resident = (size_t)std::max(1, cus) * one_dim_blocks_per_cu();
  // integrals per unit: as many as still give every resident block one
  const uint32_t per =
      (uint32_t)std::min<size_t>(kOneDimMaxUnit, std::max<size_t>(1, total / resident));
  std::vector<OneDimUnit> units;
  units.reserve(total / per + groups.size());
  for (size_t g = 0; g < groups.size(); ++g)
    for (uint32_t i = 0; i < groups[g].count; i += per)
      units.push_back(OneDimUnit{(uint32_t)g, i, std::min(per, groups[g].count - i)});
  // one upload: outcome words, groups, jobs, units; the retry list behind them
  struct Outcome {
    unsigned long long failed;
    uint32_t nretry, pad;
  };
  auto al = [](size_t x) { return (x + 255) & ~size_t(255); };
  const size_t o_groups = al(sizeof(Outcome));
  const size_t o_jobs = al(o_groups + groups.size() * sizeof(OneDimGroup));
  const size_t o_units = al(o_jobs + jobs.size() * sizeof(OneDimJob));
  const size_t o_retry = al(o_units + units.size() * sizeof(OneDimUnit));
  const uint32_t blocks = (uint32_t)std::min(units.size(), resident);
  int rc;
  if ((rc = c->od_in.ensure(o_retry + total * sizeof(OneDimUnit)))) return rc;
  // the top of the groups' trees as tables, where several blocks would work
  // them out for themselves
  const bool top = !precomp && 2 * groups.size() <= blocks;
  // nodes per block: an integral alone in a block mostly needs fewer than 2048,
  // all of a precomputation's about 300 (those that need more are refined again
  // below); a small store keeps a context's first run cheap to allocate
  const uint32_t nodes = precomp ? 1024 : per == 1 ? 2048 : kOneDimNodes;
  const size_t solo = one_dim_store_bytes(kOneDimNodes, 1);   // of a block of the second launch
  const size_t store_bytes = std::max(blocks * one_dim_store_bytes(nodes, per), solo);
  if ((rc = c->od_store.ensure(store_bytes + (top ? groups.size() * one_dim_top_bytes() : 0))))
    return rc;
  std::vector<unsigned char> host(o_retry, 0);
  Outcome oc{~0ull, 0, 0};
  std::memcpy(host.data(), &oc, sizeof(oc));
  std::memcpy(host.data() + o_groups, groups.data(), groups.size() * sizeof(OneDimGroup));
  std::memcpy(host.data() + o_jobs, jobs.data(), jobs.size() * sizeof(OneDimJob));
  std::memcpy(host.data() + o_units, units.data(), units.size() * sizeof(OneDimUnit));
  unsigned char *base = c->od_in.as<unsigned char>();
  hipStream_t s = c->stream;
  G3L_HIP(hipMemcpyAsync(base, host.data(), host.size(), hipMemcpyHostToDevice, s));
  OneDimLaunch L{};
  L.T = c->T;
  L.groups = reinterpret_cast<const OneDimGroup *>(base + o_groups);
  L.jobs = reinterpret_cast<const OneDimJob *>(base + o_jobs);
  L.units = reinterpret_cast<const OneDimUnit *>(base + o_units);
  L.nunits = (uint32_t)units.size();
  L.reltol = reltol;
  L.scale = scale;
  L.store = c->od_store.as<unsigned char>();
  L.store_bytes = one_dim_store_bytes(nodes, per);
  L.nodes = nodes;
  L.waves = per;
  L.top = top ? L.store + store_bytes : nullptr;
  L.retry = reinterpret_cast<OneDimUnit *>(base + o_retry);
  L.failed = reinterpret_cast<unsigned long long *>(base);
  L.nretry = reinterpret_cast<uint32_t *>(base + offsetof(Outcome, nretry));
  if (top) G3L_HIP(launch_one_dim_top(L, (uint32_t)groups.size(), s));
  G3L_HIP(launch_one_dim(precomp, L, blocks, s));
  G3L_HIP(hipMemcpyAsync(&oc, base, sizeof(oc), hipMemcpyDeviceToHost, s));
  G3L_HIP(hipStreamSynchronize(s));
  if (oc.nretry) {
    // integrals whose block ran out of nodes, each alone in a block with room
    // for all it can need: no more retries
    const uint32_t sb = (uint32_t)std::min<size_t>(
        {(size_t)oc.nretry, resident, store_bytes / solo});
    L.units = L.retry;
    L.nunits = oc.nretry;
    L.store_bytes = solo;
    L.nodes = kOneDimNodes;
    L.waves = 1;
    G3L_HIP(launch_one_dim(precomp, L, sb, s));
    G3L_HIP(hipMemcpyAsync(&oc, base, sizeof(oc), hipMemcpyDeviceToHost, s));
    G3L_HIP(hipStreamSynchronize(s));
  }
  return oc.failed == ~0ull ? (int)G3L_OK : status_of((uint32_t)(oc.failed & 0xff));
}

int run_one_dim(g3l_ctx *c, const std::vector<OneDimGroup> &groups,
                const std::vector<OneDimJob> &jobs, bool precomp, double reltol, double scale) {
  std::vector<OneDimGroup> part;
  size_t n = 0;
  for (const OneDimGroup &g : groups)
    for (uint32_t first = 0; first < g.count;) {
      OneDimGroup p = g;
      p.count = (uint32_t)std::min<size_t>(g.count - first, kOneDimBatch - n);
      p.job0 += first;
      p.out += first;
      first += p.count;
      n += p.count;
      part.push_back(p);
      if (n < kOneDimBatch) continue;
      if (int rc = run_one_dim_batch(c, part, jobs, precomp, reltol, scale)) return rc;
      part.clear();
      n = 0;
    }
  return n ? run_one_dim_batch(c, part, jobs, precomp, reltol, scale) : (int)G3L_OK;
}

}  // namespace g3l

namespace {

// ---------------------------------------------------------------------------
// Plain engine: the reference's driver (src/hcubature.cpp:904-1021) on the
// host, each batch of regions evaluated by one k_eval launch.
//
// Regions live in one array and stay where they are; the heap holds their keys
// and indices.  Halves go to the device as they are made: every kPlainChunk of
// them are one launch, which reads their geometry from pinned host memory and
// writes values, errors and split dimensions back there, while the host takes the
// next regions off the heap.  A triplet's three integrals (54037 regions) 16.0 ms
// with 170-byte regions moved through the heap, three copies per batch and the
// host waiting, 6.7 now.
struct HRegion {
  double c[kMaxDim], h[kMaxDim];
  double vol, val, err;
  int split;
};
// Small enough that the first launch of a large batch goes out early, large enough
// to fill the chip: 512, 1024, 2048 regions 7.3, 6.9, 6.7 ms for the three above.
constexpr size_t kPlainChunk = 2048;
// Most regions in pinned memory; beyond, the host waits and starts over in it.
constexpr size_t kPlainMax = 32768;
// The fields' rows are kept out of step with the host's caches.
constexpr size_t kPlainPad = 24;

double box_volume(int D, const double *h) {
  double v = 1;
  for (int i = 0; i < D; ++i) v *= 2 * h[i];
  return v;
}

void cut(int D, HRegion &R, HRegion &R2) {
  int d = R.split;
  R2 = R;
  R.h[d] *= 0.5;
  R.vol *= 0.5;
  for (int i = 0; i < D; ++i) {
    R2.c[i] = R.c[i];
    R2.h[i] = R.h[i];
  }
  R2.vol = box_volume(D, R2.h);
  R.c[d] -= R.h[d];
  R2.c[d] += R.h[d];
}

// The reference's heap (its comparisons, in its order) over region indices.
struct HHeap {
  struct Entry {
    double key;
    uint32_t id;
  };
  std::vector<Entry> a;
  double tval = 0, terr = 0;
  void push(uint32_t id, const HRegion &r) {
    tval += r.val;
    terr += r.err;
    const double key = r.err > 0 ? r.err : 0;
    size_t at = a.size();
    a.push_back(Entry{key, id});
    while (at) {
      size_t parent = (at - 1) / 2;
      if (key <= a[parent].key) break;
      a[at] = a[parent];
      at = parent;
    }
    a[at] = Entry{key, id};
  }
  // The last entry sinks from the root past every larger child.  It mostly ends
  // near the leaves, so the hole goes all the way down first, without a
  // comparison to mispredict, and the entry climbs back.
  uint32_t pop(const std::vector<HRegion> &regions) {
    const uint32_t top = a[0].id;
    const Entry x = a.back();
    a.pop_back();
    const size_t n = a.size();
    if (n) {
      size_t i = 0, child = 2;
      for (; child < n; child = 2 * i + 2) {
        child -= !(a[child - 1].key < a[child].key);
        a[i] = a[child];
        i = child;
      }
      if (child == n) {
        a[i] = a[n - 1];
        i = n - 1;
      }
      while (i) {
        const size_t parent = (i - 1) / 2;
        if (!(a[parent].key <= x.key)) break;
        a[i] = a[parent];
        i = parent;
      }
      a[i] = x;
      const char *next = reinterpret_cast<const char *>(&regions[a[0].id]);
      for (size_t b = 0; b < sizeof(HRegion); b += 64) __builtin_prefetch(next + b);
    }
    tval -= regions[top].val;
    terr -= regions[top].err;
    return top;
  }
};

int plain_ensure(g3l_ctx *c, uint32_t cap) {
  if (cap <= c->pcap) return G3L_OK;
  int rc;
  if ((rc = c->plist.ensure((size_t)cap * sizeof(EvalItem)))) return rc;
  if ((rc = c->hgeo.ensure((cap + kPlainPad) * kNumFields * sizeof(double)))) return rc;
  if ((rc = c->hsplit.ensure(cap))) return rc;
  std::vector<EvalItem> ident(cap);
  for (uint32_t i = 0; i < cap; ++i) ident[i] = EvalItem{i, 0};
  G3L_HIP(hipMemcpy(c->plist.p, ident.data(), cap * sizeof(EvalItem), hipMemcpyHostToDevice));
  c->pcap = cap;
  return G3L_OK;
}

// Regions on their way through the device: add() each, then finish() before their
// values are read.
struct PlainEval {
  g3l_ctx *c;
  int kind, D;
  std::vector<HRegion> &R;
  std::vector<uint32_t> ids;   // of the regions in pinned memory
  size_t sent = 0;             // of these, in launches

  // after an error, launches may still be reading the buffers
  ~PlainEval() {
    if (sent) (void)hipStreamSynchronize(c->stream);
  }
  int send() {
    if (sent == ids.size()) return G3L_OK;
    void *geo = nullptr, *split = nullptr;
    G3L_HIP(hipHostGetDevicePointer(&geo, c->hgeo.p, 0));
    G3L_HIP(hipHostGetDevicePointer(&split, c->hsplit.p, 0));
    EvalLaunch EL{};
    EL.T = c->T;
    EL.args = c->parg.as<TermArgs>();
    EL.jobs = c->pjob.as<JobDesc>();
    EL.list = c->plist.as<EvalItem>() + sent;
    EL.count = (uint32_t)(ids.size() - sent);
    EL.geo = static_cast<double *>(geo);
    EL.split = static_cast<uint8_t *>(split);
    EL.stride = c->pcap + kPlainPad;
    EL.njobs = 1;
    G3L_HIP(launch_eval(kind, G3L_FP64, c->variant[0][kind], EL, c->stream));
    sent = ids.size();
    return G3L_OK;
  }
  int finish() {
    if (int rc = send()) return rc;
    G3L_HIP(hipStreamSynchronize(c->stream));
    const size_t St = c->pcap + kPlainPad;
    const double *val = c->hgeo.as<double>() + kFieldVal * St;
    const double *err = c->hgeo.as<double>() + kFieldErr * St;
    const uint8_t *split = c->hsplit.as<uint8_t>();
    for (size_t i = 0; i < ids.size(); ++i) {
      HRegion &r = R[ids[i]];
      r.val = val[i];
      r.err = err[i];
      r.split = split[i];
    }
    ids.clear();
    sent = 0;
    return G3L_OK;
  }
  int add(uint32_t id) {
    int rc;
    if (ids.size() == c->pcap) {
      if ((rc = finish())) return rc;
      const size_t cap = c->pcap ? 2 * (size_t)c->pcap : 4096;
      if (cap <= kPlainMax && (rc = plain_ensure(c, (uint32_t)cap))) return rc;
    }
    const HRegion &r = R[id];
    const size_t St = c->pcap + kPlainPad;
    double *g = c->hgeo.as<double>() + ids.size();
    for (int d = 0; d < D; ++d) {
      g[(kFieldC + d) * St] = r.c[d];
      g[(kFieldH + d) * St] = r.h[d];
    }
    g[kFieldVol * St] = r.vol;
    ids.push_back(id);
    return ids.size() - sent == kPlainChunk ? send() : G3L_OK;
  }
};

bool converged(double val, double err, double reltol) {
  return !(err > 0 && err > std::fabs(val) * reltol);
}

int plain_cubature(g3l_ctx *c, int kind, const double *lo, const double *hi, uint64_t maxEval,
                   double reltol, double *val, double *err, uint64_t *neval, uint32_t *rounds,
                   bool *capped) {
  const int D = kind_dim(kind);
  const int np = rule_points(D);
  HRegion root{};
  for (int i = 0; i < D; ++i) {
    root.c[i] = 0.5 * (lo[i] + hi[i]);
    root.h[i] = 0.5 * (hi[i] - lo[i]);
  }
  root.vol = box_volume(D, root.h);
  std::vector<HRegion> R;
  R.reserve(kPlainMax);
  R.push_back(root);
  std::vector<uint32_t> batch;
  PlainEval E{c, kind, D, R, {}};
  uint64_t numEval = 0;
  uint32_t nb = 0;
  HHeap heap;
  int rc;
  if ((rc = E.add(0)) || (rc = E.finish())) return rc;
  ++nb;
  heap.push(0, R[0]);
  numEval += np;
  *capped = false;
  while (numEval < maxEval || !maxEval) {
    if (converged(heap.tval, heap.terr, reltol)) break;
    batch.clear();
    double eval_ = heap.tval, eerr = heap.terr;
    do {
      const uint32_t p = heap.pop(R), q = (uint32_t)R.size();
      eerr -= R[p].err;
      R.emplace_back();
      cut(D, R[p], R[q]);
      batch.push_back(p);
      batch.push_back(q);
      if ((rc = E.add(p)) || (rc = E.add(q))) return rc;
      numEval += (uint64_t)np * 2;
      if (converged(eval_, eerr, reltol)) break;
    } while (!heap.a.empty() && (numEval < maxEval || !maxEval));
    if ((rc = E.finish())) return rc;
    ++nb;
    for (uint32_t i : batch) heap.push(i, R[i]);
  }
  if (maxEval && numEval >= maxEval) *capped = true;
  double v = 0, e = 0;
  for (const HHeap::Entry &t : heap.a) {
    v += R[t.id].val;
    e += R[t.id].err;
  }
  *val = v;
  *err = e;
  *neval = numEval;
  *rounds = nb;
  return G3L_OK;
}

// n_bar(z_i) = ln10 * int m n(m,z) (Ncen + Nsat) dlog10 m for every grid z
// and both HODs of each new set (src/NNMap_Model.cu:244-282), all on the
// device in one run.
int compute_nbar(g3l_ctx *c, int first, int count) {
  const int nb = c->nb;
  const size_t need_chunks = ((size_t)first + count + kSetsPerChunk - 1) / kSetsPerChunk;
  while (c->nbar_chunks.size() < need_chunks) {
    NbarChunk b;
    b.host.resize((size_t)kSetsPerChunk * 2 * nb);
    int rc = b.dev.ensure(b.host.size() * sizeof(double));
    if (rc) return rc;
    c->nbar_chunks.push_back(std::move(b));
  }
  std::vector<OneDimJob> zs(nb);
  for (int i = 0; i < nb; ++i) zs[i] = OneDimJob{c->zmin + i * (c->zmax - c->zmin) / nb, 0, 0};
  std::vector<OneDimGroup> groups;
  groups.reserve(2 * (size_t)count);
  for (int s = first; s < first + count; ++s)
    for (int which = 0; which < 2; ++which) {
      OneDimGroup g{};
      g.h = to_dev(which == 0 ? c->sets[s].h1 : c->sets[s].h2);
      g.rs = 1. / g.h.sigma;
      g.lo = std::log10(c->mmin_i);
      g.hi = std::log10(c->mmax_i);
      g.out = const_cast<double *>(nbar_ptr(c, s, which));
      g.count = (uint32_t)nb;
      g.mode = kOneDNbar;
      groups.push_back(g);
    }
  if (int rc = run_one_dim(c, groups, zs, false, 1e-4, kLn10)) return rc;
  // one copy per storage chunk that the sets touch
  for (int s = first; s < first + count;) {
    const int e = std::min(first + count, (s / kSetsPerChunk + 1) * kSetsPerChunk);
    const size_t at = (size_t)(s % kSetsPerChunk) * 2 * nb;
    G3L_HIP(hipMemcpyAsync(c->nbar_chunks[s / kSetsPerChunk].host.data() + at, nbar_ptr(c, s, 0),
                           (size_t)(e - s) * 2 * nb * sizeof(double), hipMemcpyDeviceToHost,
                           c->stream));
    s = e;
  }
  G3L_HIP(hipStreamSynchronize(c->stream));
  return G3L_OK;
}

}  // namespace

// ===========================================================================
// C ABI
extern "C" {

const char *g3l_version(void) { return "g3lhalo_amd 0.1 (gfx950)"; }

int g3l_ctx_create(const g3l_tables *t, g3l_ctx **out) {
  if (!t || !out || t->nbins < 2 || t->nbins > 46340 || !t->g || !t->p_lens1 || !t->w ||
      !t->dwdz || !t->hmf ||
      !t->P_lin || !t->b_h || !t->concentration)
    return G3L_EINVAL;
  if (!(t->zmax > t->zmin) || !(t->kmax > t->kmin) || !(t->mmax > t->mmin) || t->mmin <= 0 ||
      t->kmin <= 0)
    return G3L_EINVAL;
  g3l_ctx *c = nullptr;
  if (int rc = ctx_create_bare(&c)) return rc;
  const int nb = t->nbins;
  c->nb = nb;
  c->zmin = t->zmin; c->zmax = t->zmax; c->kmin = t->kmin; c->kmax = t->kmax;
  c->mmin = t->mmin; c->mmax = t->mmax;
  c->H0 = t->H0; c->Om = t->Omega_m; c->OL = t->Omega_Lambda;
  c->rho_crit = 3 * c->H0 * c->H0 * kMpcKm / 8 / kPi / kGMsun;
  // integral borders (src/NNMap_Model.cu:46-49)
  c->zmin_i = c->zmin;
  c->zmax_i = c->zmax - (c->zmax - c->zmin) / nb;
  c->mmin_i = c->mmin;
  c->mmax_i = std::exp(std::log(c->mmin) + std::log(c->mmax / c->mmin) * (nb - 1) / nb);
  // rho_bar(z) = Omega_m(z) rho_crit (src/NNMap_Model.cu:256, src/Cosmology.cpp:79-87)
  c->rho.resize(nb);
  for (int i = 0; i < nb; ++i) {
    double z = c->zmin + i * (c->zmax - c->zmin) / nb;
    double E = c->Om * (1 + z) * (1 + z) * (1 + z) + c->OL;
    c->rho[i] = c->Om * (1 + z) * (1 + z) * (1 + z) / E * c->rho_crit;
  }
  const size_t n1 = nb, n2 = (size_t)nb * nb;
  const size_t total = 8 * n1 + 4 * n2 + n1 + DevTables::kConsts;
  if (c->tables.ensure(total * sizeof(double))) {
    g3l_ctx_destroy(c);
    return G3L_ENOMEM;
  }
  std::vector<double> h(total, 0.0);
  double *p = h.data();
  auto put = [&](const double *src, size_t n) {
    double *at = p;
    if (src) std::memcpy(p, src, n * sizeof(double));
    p += n;
    return (size_t)(at - h.data());
  };
  std::vector<double> rw(nb), rrho(nb);
  for (int i = 0; i < nb; ++i) {
    rw[i] = 1. / t->w[i];
    rrho[i] = 1. / c->rho[i];
  }
  const long double lmm = std::log((long double)c->mmin);
  double lo[kMaxDim], hi[kMaxDim];
  term_box(c, 1, lo, hi);
  double consts[DevTables::kConsts] = {(double)lmm, (double)(lmm - (double)lmm),
                                       0.5 * (lo[3] + hi[3])};
  const size_t orw = put(rw.data(), n1), orr = put(rrho.data(), n1),
               oconst = put(consts, DevTables::kConsts);
  size_t og = put(t->g, n1), op1 = put(t->p_lens1, n1),
         op2 = put(t->p_lens2 ? t->p_lens2 : t->p_lens1, n1), ow = put(t->w, n1),
         odw = put(t->dwdz, n1), orho = put(c->rho.data(), n1), ohmf = put(t->hmf, n2),
         opl = put(t->P_lin, n2);
  // P_lin keeps nb trailing zeros (h is zero-filled; the caller's array has
  // n2 entries): the look-up has no upper guard (src/NNMap_Model.cu:826-839),
  // so the last row's overrun reads zeros.
  put(nullptr, n1);
  size_t obh = put(t->b_h, n2), oc = put(t->concentration, n2);
  if (hipMemcpy(c->tables.p, h.data(), total * sizeof(double), hipMemcpyHostToDevice) !=
      hipSuccess) {
    g3l_ctx_destroy(c);
    return G3L_EHIP;
  }
  double *d = c->tables.as<double>();
  DevTables &T = c->T;
  T.nb = nb;
  T.zmin = c->zmin; T.zmax = c->zmax; T.kmin = c->kmin; T.kmax = c->kmax;
  T.mmin = c->mmin; T.mmax = c->mmax;
  T.lmr = std::log(c->mmax / c->mmin);
  T.lkr = std::log(c->kmax / c->kmin);
  T.rdz = 1. / (c->zmax - c->zmin);
  T.rkmin = 1. / c->kmin;
  T.rlkr = 1. / T.lkr;
  T.rmmin = 1. / c->mmin;
  T.rlmr = 1. / T.lmr;
  T.rw = d + orw;
  T.rrho = d + orr;
  T.g = d + og; T.p1 = d + op1; T.p2 = d + op2; T.w = d + ow; T.dwdz = d + odw;
  T.rho = d + orho; T.hmf = d + ohmf; T.plin = d + opl; T.bh = d + obh; T.conc = d + oc;
  if (launch_mass_centre(T, d + oconst + 3, c->stream) != hipSuccess ||
      hipStreamSynchronize(c->stream) != hipSuccess) {
    g3l_ctx_destroy(c);
    return G3L_EHIP;
  }
  *out = c;
  return G3L_OK;
}

int g3l_ctx_destroy(g3l_ctx *c) {
  if (!c) return G3L_EINVAL;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  c->tables.release();
  for (auto &b : c->nbar_chunks) b.dev.release();
  c->nbar_chunks.clear();
  c->pool.release(); c->split.release(); c->lists.release(); c->jobs.release();
  c->state.release(); c->args.release(); c->boxes.release(); c->counters.release();
  c->hcounters.release();
  c->trace.release();
  c->od_store.release(); c->od_in.release();
  c->plist.release(); c->pjob.release();
  c->parg.release(); c->hgeo.release(); c->hsplit.release();
  for (auto &e : c->ev)
    if (e) (void)hipEventDestroy(e);
  for (auto &e : c->kev)
    if (e) (void)hipEventDestroy(e);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  return G3L_OK;
}

int g3l_hodset_create_many(g3l_ctx *c, int32_t n, const g3l_hod *hod1, const g3l_hod *hod2,
                           const double *A, const double *eps, const int32_t *identical,
                           int32_t *first_id) {
  if (!c || n <= 0 || !hod1 || !first_id) return G3L_EINVAL;
  int first = (int)c->sets.size();
  for (int i = 0; i < n; ++i) {
    HodSet s;
    s.h1 = hod1[i];
    s.h2 = hod2 ? hod2[i] : hod1[i];
    s.A = A ? A[i] : 0.0;
    s.eps = eps ? eps[i] : 0.0;
    s.identical = identical ? identical[i] : 0;
    for (const g3l_hod *h : {&s.h1, &s.h2})
      if (!(h->mth > 0) || !(h->sigma > 0) || !(h->mprime > 0)) {
        c->sets.resize(first);
        return G3L_EINVAL;
      }
    c->sets.push_back(s);
  }
  int rc = compute_nbar(c, first, n);
  if (rc) {
    c->sets.resize(first);
    return rc;
  }
  *first_id = first;
  return G3L_OK;
}

int g3l_hodset_create(g3l_ctx *c, const g3l_hod *hod1, const g3l_hod *hod2, double A,
                      double epsilon, int32_t identical, int32_t *set_id) {
  return g3l_hodset_create_many(c, 1, hod1, hod2, &A, &epsilon, &identical, set_id);
}

int g3l_hodset_densities(g3l_ctx *c, int32_t set, double *rho_bar, double *n_bar1,
                         double *n_bar2) {
  if (!c || set < 0 || set >= (int)c->sets.size()) return G3L_EINVAL;
  if (rho_bar) std::memcpy(rho_bar, c->rho.data(), c->nb * sizeof(double));
  const double *h = c->nbar_chunks[set / kSetsPerChunk].host.data() +
                    (size_t)(set % kSetsPerChunk) * 2 * c->nb;
  if (n_bar1) std::memcpy(n_bar1, h, c->nb * sizeof(double));
  if (n_bar2) std::memcpy(n_bar2, h + c->nb, c->nb * sizeof(double));
  return G3L_OK;
}

int g3l_hodset_clear(g3l_ctx *c) {
  if (!c) return G3L_EINVAL;
  c->sets.clear();
  return G3L_OK;
}

int g3l_eval_plain(g3l_ctx *c, const g3l_request *r, g3l_result *out) {
  if (!c || !r || !out) return G3L_EINVAL;
  int rc = check_request(c, *r);
  if (rc) return rc;
  const int kind = kind_of(r->stat, r->term);
  TermArgs a = make_args(c, *r);
  JobDesc d{};
  d.kind = kind;
  d.dim = kind_dim(kind);
  d.pts = rule_points(d.dim);
  d.args = 0;
  if ((rc = c->parg.ensure(sizeof(TermArgs)))) return rc;
  if ((rc = c->pjob.ensure(sizeof(JobDesc)))) return rc;
  G3L_HIP(hipMemcpy(c->parg.p, &a, sizeof(a), hipMemcpyHostToDevice));
  G3L_HIP(hipMemcpy(c->pjob.p, &d, sizeof(d), hipMemcpyHostToDevice));
  double lo[kMaxDim], hi[kMaxDim];
  term_box(c, r->term, lo, hi);
  double val = 0, err = 0;
  uint64_t ne = 0;
  uint32_t nbt = 0;
  bool capped = false;
  rc = plain_cubature(c, kind, lo, hi, r->maxeval, r->reltol, &val, &err, &ne, &nbt, &capped);
  if (rc) return rc;
  out->raw = val;
  out->err = err;
  out->value = prefactor(c, r->stat, r->term, val);
  out->neval = ne;
  out->rounds = nbt;
  out->status = !std::isfinite(val) || !std::isfinite(err) ? G3L_NONFINITE
                : capped                                     ? G3L_MAXEVAL_HIT
                                                             : G3L_OK;
  return G3L_OK;
}

int g3l_eval_batch(g3l_ctx *c, const g3l_request *reqs, size_t n, int32_t precision,
                   g3l_result *out) {
  if (!c || (!reqs && n) || (!out && n)) return G3L_EINVAL;
  if (precision != G3L_FP64 && precision != G3L_MIXED) return G3L_EINVAL;
  EngineJobs E;
  E.desc.reserve(n);
  E.args.reserve(n);
  E.boxes.reserve(n * 2 * kMaxDim);
  for (size_t i = 0; i < n; ++i) {
    int rc = check_request(c, reqs[i]);
    if (rc) return rc;
    const int kind = kind_of(reqs[i].stat, reqs[i].term);
    JobDesc d{};
    d.kind = kind;
    d.dim = kind_dim(kind);
    d.pts = rule_points(d.dim);
    d.args = (int)i;
    d.reltol = reqs[i].reltol;
    d.maxeval = reqs[i].maxeval;
    d.cap = slot_cap(d.maxeval, d.pts, 1u << 16);
    E.desc.push_back(d);
    E.args.push_back(make_args(c, reqs[i]));
    double box[2 * kMaxDim] = {0};
    term_box(c, reqs[i].term, box, box + kMaxDim);
    E.boxes.insert(E.boxes.end(), box, box + 2 * kMaxDim);
  }
  std::vector<JobState> st;
  int rc = run_engine(c, E, st, true, precision, true);
  if (rc) return rc;
  for (size_t i = 0; i < n; ++i) {
    out[i].raw = st[i].val;
    out[i].err = st[i].err;
    out[i].value = prefactor(c, reqs[i].stat, reqs[i].term, st[i].val);
    out[i].neval = st[i].neval;
    out[i].rounds = st[i].rounds + 1;
    out[i].status = status_of(st[i].flags);
  }
  return G3L_OK;
}


int g3l_integrand(g3l_ctx *c, const g3l_request *r, int32_t precision, size_t npts,
                  const double *x, double *f) {
  if (!c || !r || (npts && (!x || !f)) || npts > 0xffffffffull) return G3L_EINVAL;
  if (precision != G3L_FP64 && precision != G3L_MIXED) return G3L_EINVAL;
  int rc;
  int kind;
  TermArgs a{};
  if (r->term == 0) {
    if (r->hodset < 0 || r->hodset >= (int)c->sets.size()) return G3L_EINVAL;
    kind = kNbar;
    a.t1 = r->theta[0];
    const HodSet &s = c->sets[r->hodset];
    a.h1 = a.h2 = to_dev(r->type1 == 2 ? s.h2 : s.h1);
    a.rs1 = a.rs2 = 1. / a.h1.sigma;
    fill_logs(c, a);
  } else {
    if ((rc = check_request(c, *r))) return rc;
    kind = kind_of(r->stat, r->term);
    a = make_args(c, *r);
  }
  if (npts == 0) return G3L_OK;
  const int D = kind_dim(kind);
  DevBuf dx, df, da;
  if (dx.ensure(npts * D * sizeof(double)) || df.ensure(npts * sizeof(double)) ||
      da.ensure(sizeof(TermArgs))) {
    dx.release(); df.release(); da.release();
    return G3L_ENOMEM;
  }
  rc = G3L_OK;
  if (hipMemcpy(dx.p, x, npts * D * sizeof(double), hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(da.p, &a, sizeof(a), hipMemcpyHostToDevice) != hipSuccess ||
      launch_points(kind, precision, c->T, da.as<TermArgs>(), dx.as<double>(), (uint32_t)npts,
                    df.as<double>(), c->stream) != hipSuccess ||
      hipStreamSynchronize(c->stream) != hipSuccess ||
      hipMemcpy(f, df.p, npts * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
    rc = G3L_EHIP;
  dx.release(); df.release(); da.release();
  return rc;
}

int g3l_set_trace(g3l_ctx *c, uint32_t cap) {
  if (!c || cap > 4096) return G3L_EINVAL;
  c->trace_cap = cap;
  c->trace_jobs = 0;
  c->trace_rounds.clear();
  return G3L_OK;
}

int g3l_last_trace(g3l_ctx *c, size_t i, uint32_t *regions, uint32_t cap, uint32_t *len) {
  if (!c || !len || (cap && !regions)) return G3L_EINVAL;
  if (c->trace_cap == 0 || i >= c->trace_jobs) return G3L_EINVAL;
  const uint32_t rounds = c->trace_rounds[i] + 1;  // the root's evaluation included
  uint32_t n = std::min<uint32_t>(std::min<uint32_t>(rounds, c->trace_cap + 1), cap);
  if (n > 0) {
    regions[0] = 1;
    if (n > 1)
      G3L_HIP(hipMemcpy(regions + 1, c->trace.as<uint32_t>() + i * c->trace_cap,
                        (n - 1) * sizeof(uint32_t), hipMemcpyDeviceToHost));
  }
  *len = n;
  return G3L_OK;
}

int g3l_last_batch_stats(g3l_ctx *c, g3l_batch_stats *out) {
  if (!c || !out) return G3L_EINVAL;
  *out = c->last;
  return G3L_OK;
}

int g3l_autotune(g3l_ctx *c, int32_t hodset, int32_t precision, g3l_tune_report *out) {
  if (!c || hodset < 0 || hodset >= (int)c->sets.size()) return G3L_EINVAL;
  if (precision != G3L_FP64 && precision != G3L_MIXED) return G3L_EINVAL;
  // calibration: 55 aperture triplets x 1h/2h/3h for each statistic, at the
  // production tolerance and budget (launch sizes like the real workloads)
  const double arcmin = 2.909e-4;
  std::vector<g3l_request> reqs[2];
  for (int st = 0; st < 2; ++st)
    for (int i = 0; i < 55; ++i) {
      const int a = i % 10, b = (i * 3) % 10, d = (i * 7) % 10;
      for (int term = 1; term <= 3; ++term) {
        g3l_request r{};
        r.stat = st;
        r.term = term;
        r.hodset = hodset;
        r.type1 = 1;
        r.type2 = 2;
        r.theta[0] = 0.5 * std::pow(64.0, a / 9.0) * arcmin;
        r.theta[1] = 0.5 * std::pow(64.0, b / 9.0) * arcmin;
        r.theta[2] = 0.5 * std::pow(64.0, d / 9.0) * arcmin;
        r.reltol = 1e-4;
        r.maxeval = 5000000;
        reqs[st].push_back(r);
      }
    }
  const int pi = precision == G3L_MIXED;
  const int nv = eval_num_variants();
  double ms[kNumKinds][8] = {};
  const g3l_batch_stats keep = c->last;
  for (int v = 0; v < nv && v < 8; ++v) {
    for (int k = 1; k < kNumKinds; ++k) c->variant[pi][k] = v;
    for (int st = 0; st < 2; ++st) {
      EngineJobs E;
      for (const g3l_request &r : reqs[st]) {
        const int kind = kind_of(r.stat, r.term);
        JobDesc d{};
        d.kind = kind;
        d.dim = kind_dim(kind);
        d.pts = rule_points(d.dim);
        d.args = (int)E.args.size();
        d.reltol = r.reltol;
        d.maxeval = r.maxeval;
        d.cap = slot_cap(d.maxeval, d.pts, 1u << 16);
        E.desc.push_back(d);
        E.args.push_back(make_args(c, r));
        double box[2 * kMaxDim] = {0};
        term_box(c, r.term, box, box + kMaxDim);
        E.boxes.insert(E.boxes.end(), box, box + 2 * kMaxDim);
      }
      std::vector<JobState> jst;
      for (int rep = 0; rep < 2; ++rep) {  // the first run warms up
        int rc = run_engine(c, E, jst, true, precision);
        if (rc) {
          c->last = keep;
          return rc;
        }
      }
      for (int k = 1; k < kNumKinds; ++k) ms[k][v] += c->last.kind_ms[k];
    }
  }
  c->last = keep;
  for (int k = 1; k < kNumKinds; ++k) {
    int best = 0;
    for (int v = 1; v < nv; ++v)
      if (ms[k][v] < ms[k][best]) best = v;
    c->variant[pi][k] = best;
  }
  if (out) {
    *out = g3l_tune_report{};
    for (int k = 0; k < kNumKinds && k < 8; ++k) {
      out->variant[k] = c->variant[pi][k];
      for (int v = 0; v < nv && v < 4; ++v) {
        out->ms[k][v] = ms[k][v];
        out->group[k][v] = eval_group_size(k, v);
      }
    }
  }
  return G3L_OK;
}

int g3l_set_launch_mode(g3l_ctx *c, int32_t mode) {
  if (!c || (mode != G3L_LAUNCH_STREAM && mode != G3L_LAUNCH_GRAPH)) return G3L_EINVAL;
  c->launch_mode = mode;
  return G3L_OK;
}

int g3l_set_mixed_policy(g3l_ctx *c, uint32_t fp32_kinds) {
  if (!c || (fp32_kinds & ~0x7eu)) return G3L_EINVAL;  // kinds 1-6 only
  c->mixed_fp32_kinds = fp32_kinds;
  return G3L_OK;
}

int g3l_get_mixed_policy(g3l_ctx *c, uint32_t *fp32_kinds) {
  if (!c || !fp32_kinds) return G3L_EINVAL;
  *fp32_kinds = c->mixed_fp32_kinds;
  return G3L_OK;
}

int g3l_set_variant(g3l_ctx *c, int32_t kind, int32_t precision, int32_t variant) {
  if (!c || kind < 1 || kind >= kNumKinds || variant < 0 || variant >= eval_num_variants())
    return G3L_EINVAL;
  if (precision != G3L_FP64 && precision != G3L_MIXED) return G3L_EINVAL;
  c->variant[precision == G3L_MIXED][kind] = variant;
  return G3L_OK;
}

}  // extern "C"
