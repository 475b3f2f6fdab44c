// One wave of 64 lanes on the host: a context per lane, taken in turn; a cross-lane
// operation leaves its lane's word and goes on once every lane has left one.  Every
// lane has to reach every operation, as in the wave functions it is for
// (select_wave.h).
#pragma once
#include <math.h>
#include <stdint.h>
#include <ucontext.h>

#define __device__
#define __host__
#define __forceinline__ inline

namespace hostwave {
inline ucontext_t lanes[64], turn;
inline int lane;                     // the one that runs
inline uint64_t word[2][64];
inline unsigned step[64];            // operations of each lane
// every lane's v
inline const uint64_t *gather(uint64_t v) {
  uint64_t *w = word[step[lane]++ & 1];   // the other row may still be read
  w[lane] = v;
  swapcontext(&lanes[lane], &turn);
  return w;
}
// lane l's v (its own where there is no such lane)
inline uint64_t from(uint64_t v, int l) {
  const uint64_t r = gather(v)[l >= 0 && l < 64 ? l : lane];
  return r;
}
inline char stacks[64][1 << 16];
// f() once in every lane
inline void run(void (*f)()) {
  bool more[64];
  static void (*body)();
  static bool *left;
  body = f;
  left = more;
  auto start = [] {
    body();
    left[lane] = false;
    swapcontext(&lanes[lane], &turn);
  };
  for (int l = 0; l < 64; ++l) {
    more[l] = true;
    getcontext(&lanes[l]);
    lanes[l].uc_stack.ss_sp = stacks[l];
    lanes[l].uc_stack.ss_size = sizeof(stacks[l]);
    lanes[l].uc_link = nullptr;
    step[l] = 0;
    makecontext(&lanes[l], (void (*)())+start, 0);
  }
  while (more[0])
    for (lane = 0; lane < 64; ++lane)
      if (more[lane]) swapcontext(&turn, &lanes[lane]);
}
struct Index {
  operator int() const { return lane; }
};
struct Thread {
  Index x;
};
struct Pair {
  uint32_t v[2];
  uint32_t operator[](int i) const { return v[i]; }
};
}  // namespace hostwave
static hostwave::Thread threadIdx;

inline uint64_t __ballot(bool p) {
  const uint64_t *w = hostwave::gather(p);
  uint64_t m = 0;
  for (int l = 0; l < 64; ++l) m |= w[l] << l;
  return m;
}
inline int __popcll(uint64_t m) { return __builtin_popcountll(m); }
inline int __ffsll(unsigned long long m) { return __builtin_ffsll((long long)m); }
inline int __builtin_amdgcn_readlane(int v, int l) { return (int)hostwave::from((uint32_t)v, l); }
inline uint32_t __builtin_amdgcn_readfirstlane(uint32_t v) { return (uint32_t)hostwave::from(v, 0); }
inline uint32_t __builtin_amdgcn_mbcnt_lo(uint32_t m, uint32_t c) {
  return c + __builtin_popcountll(m & ((1ull << hostwave::lane) - 1));
}
inline uint32_t __builtin_amdgcn_mbcnt_hi(uint32_t m, uint32_t c) {
  return c + __builtin_popcountll(((uint64_t)m << 32) & ((1ull << hostwave::lane) - 1));
}
inline hostwave::Pair __builtin_amdgcn_permlane32_swap(uint32_t v, uint32_t, bool, bool) {
  return {{v, (uint32_t)hostwave::from(v, hostwave::lane ^ 32)}};
}
inline hostwave::Pair __builtin_amdgcn_permlane16_swap(uint32_t v, uint32_t, bool, bool) {
  return {{v, (uint32_t)hostwave::from(v, hostwave::lane ^ 16)}};
}
// row_shl: lane l of a row of 16 takes lane l + w, 0 beyond the row
inline int __builtin_amdgcn_update_dpp(int, int v, int ctrl, int, int, bool) {
  const int w = ctrl - 0x100, l = hostwave::lane;
  const uint32_t r = (uint32_t)hostwave::from((uint32_t)v, l + w);
  return (l & 15) + w < 16 ? (int)r : 0;
}
inline void __builtin_amdgcn_fence(int, const char *) { (void)hostwave::gather(0); }
inline void __builtin_amdgcn_wave_barrier() {}
