// onedim.h -- adaptive Gauss-Kronrod integrals in one dimension on the device:
// n_bar(z) of the HOD sets and the integrals of the table precomputation.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layout.h"
#include "physics.h"

namespace g3l {

// Integrals over one box [lo, hi] whose integrands share everything but the
// per-integral parameters of OneDimJob: what depends on the abscissa alone
// (one_dim_node) is computed once for all integrals a block refines together.
// Integral i of the group has the parameters jobs[job0 + i] and leaves
// scale * value in out[i].
struct OneDimGroup {
  DevHod h;              // kOneDNbar
  double rs;             // 1 / h.sigma
  double lo, hi;
  double *out;
  const double *aux;     // PrecompParams of the other modes
  uint32_t job0, count;
  int32_t mode;          // OneDMode
  int32_t pad;
};

// t1..t3 of the integrand modes (OneDMode).
struct OneDimJob {
  double t1, t2, t3;
};

// Integrals [first, first + count) of a group, refined by one block; count is
// at most kOneDimMaxUnit.
struct OneDimUnit {
  uint32_t group, first, count;
};
constexpr int kOneDimMaxUnit = 8;

// Regions an integral may hold; most nodes (regions of all its integrals, split
// ones included) a block may have room for.  An integral alone in a block with
// that much room cannot run out: 2048 regions are the leaves of a tree of 4095.
constexpr uint32_t kOneDimCap = 2048;
constexpr uint32_t kOneDimNodes = 8192;
// Nodes of a group's table of the top of its tree: twelve levels.
constexpr uint32_t kOneDimTop = 4095;

struct OneDimLaunch {
  DevTables T;                // kOneDNbar
  const OneDimGroup *groups;
  const OneDimJob *jobs;
  const OneDimUnit *units;
  uint32_t nunits;
  double reltol, scale;
  unsigned char *store;       // store_bytes per block
  size_t store_bytes;         // one_dim_store_bytes(nodes, waves)
  uint32_t nodes, waves;      // nodes a block has room for; most integrals per unit
  unsigned char *top;         // one_dim_top_bytes() per group, or null (n_bar)
  OneDimUnit *retry;          // integrals of units that ran out of nodes
  uint32_t *nretry;
  // smallest (integral's rank << 8 | job flags) over the integrals that end
  // with kJobPoolFull or kJobNonfinite; the rank orders by group, then index
  unsigned long long *failed;
};

// Device memory of one block, and of a group's table; the blocks a compute
// unit holds at a time.
size_t one_dim_store_bytes(uint32_t nodes, uint32_t waves);
size_t one_dim_top_bytes();
int one_dim_blocks_per_cu();
// Fills L.top for the groups [0, ngroups).
hipError_t launch_one_dim_top(const OneDimLaunch &L, uint32_t ngroups, hipStream_t s);
// Launches `blocks` blocks (at most L.nunits), each over a range of L.units.  precomp: the groups hold
// precomputation modes (kOneDNbar otherwise).
hipError_t launch_one_dim(bool precomp, const OneDimLaunch &L, uint32_t blocks, hipStream_t s);

}  // namespace g3l
